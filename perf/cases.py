"""The solves that users of this library run, as one-pass cases for timing and comparison.

A case is a dict of plain values:
  path     "solve"       one instance through flock_amd.solve (host arrays in and out)
           "noalloc"     the same through flock_amd.solve_noalloc
           "batch"       a resident flock_amd.Batch: one run, results read back
           "batch_solve" flock_amd.batch_solve: host arrays to complete solutions
           "server"      a flock_amd.Server: requests submitted at once, polled until done
  m, n     size of the instance; batches and servers draw `count` sizes log-uniform in [lo, hi]
  costs    "small" U{1..100}, "wide" U{1..1000}, "decimal" U{10000..99900} (two decimals, the
           range of the data files under tests/golden), "unit" U{1..8} with equal supplies and
           equal demands (the degenerate family)
  pricing, initial  the solver's options

Results.  The Dantzig rule fixes the pivot sequence, so those cases return the complete solution
(basis slot by slot, flows, duals, pivot count).  The other pricing rules promise an optimum, and
an instance can have several optimal plans: single solves use the "decimal" costs, where ties are
rare, and return the objective and the whole plan (m x n), of which a few cells may differ between
optimal plans; batches and servers under those rules return every instance's objective and status.
"""
import numpy as np

import flock_amd as F
from flock_amd import instances as I

# costs: lowest, highest, largest supply or demand drawn
COSTS = {"small": (1, 100, 1000), "wide": (1, 1000, 10000), "decimal": (10000, 99900, 1000)}


def listed():
    return [
        # the smallest call: a hand-sized instance, all launch and copy latency
        dict(name="solve_13x9_dantzig", path="solve", m=13, n=9, costs="small", pricing="dantzig", initial="vogel"),
        # the data files' usual size, with the default options
        dict(name="solve_100x100_dantzig", path="solve", m=100, n=100, costs="small", pricing="dantzig", initial="vogel"),
        # ragged and long, from a host that may not allocate, north-west corner start
        dict(name="noalloc_37x411_nwc", path="noalloc", m=37, n=411, costs="decimal", pricing="dantzig", initial="nwc"),
        # a data file of middle size, fast pricing, one workgroup
        dict(name="solve_250x490_candidates", path="solve", m=250, n=490, costs="decimal", pricing="candidates", initial="vogel"),
        # the multi-pivot / Dantzig hybrid (switchModel_parallel)
        dict(name="solve_201x150_switch", path="solve", m=201, n=150, costs="decimal", pricing="switch", initial="vogel"),
        # a 500 x 500 data file with the default options: sweep grid and rounds
        dict(name="solve_500x500_dantzig", path="solve", m=500, n=500, costs="decimal", pricing="dantzig", initial="vogel"),
        # the large single solve
        dict(name="solve_1000x1000_candidates", path="solve", m=1000, n=1000, costs="decimal", pricing="candidates", initial="vogel"),
        # the largest matrix: degenerate assignment-like costs, the initial basis dominates
        dict(name="solve_4000x2000_unit", path="solve", m=4000, n=2000, costs="unit", pricing="dantzig", initial="vogel"),
        # many small problems from host arrays to complete solutions
        dict(name="batch_solve_512_small", path="batch_solve", count=512, lo=8, hi=96, costs="small", pricing="dantzig", initial="vogel"),
        # the headline batch: instances resident, one launch
        dict(name="batch_4096_candidates", path="batch", count=4096, lo=16, hi=512, costs="small", pricing="candidates", initial="vogel"),
        # the default pricing on a resident batch that does not fill the device evenly
        dict(name="batch_300_dantzig", path="batch", count=300, lo=16, hi=400, costs="wide", pricing="dantzig", initial="vogel"),
        # a burst of requests of every size on a continuous-batching server
        dict(name="server_160_burst", path="server", count=160, lo=32, hi=2000, costs="wide", pricing="candidates", initial="vogel"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    path = rng.choice(["solve", "solve", "solve", "noalloc", "batch", "batch_solve", "server"])
    costs = rng.choice(["small", "wide", "decimal"])
    if path in ("solve", "noalloc"):
        pricing = rng.choice(["dantzig", "dantzig", "candidates", "candidates", "switch", "multi"])
        hi = {"dantzig": 700, "candidates": 1400, "switch": 300, "multi": 300}[pricing]
        lo = 4 if pricing == "dantzig" else 24
        m = _log_int(rng, lo, hi)
        n = min(_log_int(rng, lo, hi), 64 * m)  # few supplies are still enough for every demand
        initial = "nwc" if m * n <= 20000 and rng.random() < 0.25 else "vogel"
        return dict(path=path, m=m, n=n, costs=costs if pricing == "dantzig" else "decimal", pricing=pricing, initial=initial)
    pricing = rng.choice(["dantzig", "candidates"])
    lo = _log_int(rng, 4, 32)
    if path == "batch":
        return dict(path=path, count=_log_int(rng, 24, 400 if pricing == "dantzig" else 3000), lo=max(lo, 7), hi=_log_int(rng, 64, 400), costs=costs, pricing=pricing, initial="vogel")
    if path == "batch_solve":
        return dict(path=path, count=_log_int(rng, 8, 600), lo=lo, hi=_log_int(rng, 48, 160), costs=costs, pricing=pricing, initial="vogel")
    return dict(path=path, count=_log_int(rng, 16, 200), lo=max(lo, 16), hi=_log_int(rng, 100, 1000), costs=costs, pricing="candidates", initial="vogel")


def _sizes(case, rng):
    if "m" in case:
        return [(case["m"], case["n"])]
    ms = I.log_uniform_sizes(rng, case["count"], case["lo"], case["hi"])
    ns = I.log_uniform_sizes(rng, case["count"], case["lo"], case["hi"])
    return list(zip(ms.tolist(), ns.tolist()))


def _instances(case, seed):
    if case["costs"] == "unit":
        return [I.degenerate(seed, case["m"], case["n"])]
    rng = np.random.default_rng([seed, 20])
    lo, hi, amount = COSTS[case["costs"]]
    if "m" in case:
        return [I.random_instance(rng, case["m"], case["n"], hi, amount, cmin=lo)]
    # batches and bursts keep their sizes (they are the case's), the data change with the seed
    sizes = _sizes(case, np.random.default_rng([case["count"], case["lo"], case["hi"]]))
    return [I.random_instance(rng, m, n, hi, amount, cmin=lo) for m, n in sizes]


def prepare(case, seed):
    insts = _instances(case, seed)
    state = dict(case=case, insts=insts)
    if case["path"] == "batch":
        state["batch"] = F.Batch(insts)
    if case["path"] == "server":
        state["server"] = F.Server(hbm_budget_bytes=2 << 30, max_slots=512, pricing=case["pricing"], initial=case["initial"])
    return state


def _solution(case, inst, s):
    if case["pricing"] == "dantzig":
        return dict(objective=s.objective, status=s.status, iterations=s.iterations, rows=s.rows, cols=s.cols,
                    flows=s.flows, u=s.u, v=s.v)
    plan = np.zeros((inst.m, inst.n), np.int32)
    plan[s.rows, s.cols] = s.flows
    return dict(objective=s.objective, status=s.status, plan=plan)


def _totals(sols):
    return dict(objective=np.array([s.objective for s in sols], np.int64), status=np.array([s.status for s in sols], np.int32))


def _whole(sols):
    arrays = {k: np.concatenate([getattr(s, k) for s in sols]) for k in ("rows", "cols", "flows", "u", "v")}
    return dict(_totals(sols), iterations=np.array([s.iterations for s in sols], np.int64), **arrays)


def run(state):
    case, insts = state["case"], state["insts"]
    options = dict(pricing=case["pricing"], initial=case["initial"])
    if case["path"] == "solve":
        return _solution(case, insts[0], F.solve(insts[0], **options))
    if case["path"] == "noalloc":
        return _solution(case, insts[0], F.solve_noalloc(insts[0], **options))
    if case["path"] == "batch":
        state["batch"].run(**options)
        if case["pricing"] == "dantzig":
            return _whole(state["batch"].results())
        return _totals(state["batch"].results(full=False))
    if case["path"] == "batch_solve":
        sols, _ = F.batch_solve(insts, **options)
        return _whole(sols) if case["pricing"] == "dantzig" else _totals(sols)
    server = state["server"]
    tickets = [server.submit(x) for x in insts]
    done = {}
    while len(done) < len(tickets):
        done.update(server.poll(max_wait_ms=2.0, cap=256))
    return _totals([done[t] for t in tickets])


def work(case):
    """Each cost read once and compared with its duals (two subtractions and a comparison), each result written once."""
    sizes = _sizes(case, np.random.default_rng([case.get("count", 0), case.get("lo", 0), case.get("hi", 0)]))
    cells = sum(m * n for m, n in sizes)
    lines = sum(m + n for m, n in sizes)
    return dict(bytes=4 * cells + 4 * lines + 16 * lines, flops=3 * cells)


def tolerance(case):
    """Integers throughout.  Only a plan can differ at all, in the cells of a few cycles of zero reduced cost: 2.4e-5 of
    the cells between two pricing rules at 250 x 490, 2e-5 at 1000 x 1000; one cycle at 150 x 200 is about 2e-4."""
    if case["pricing"] != "dantzig" and case["path"] in ("solve", "noalloc"):
        return {"rel": 0.0, "differ": 8e-4}
    return "exact"


def _optimum(inst, limit=4000):
    """The optimal objective by the textbook method in 64 bits: north-west corner, duals, most negative reduced cost."""
    m, n = inst.m, inst.n
    cost = inst.cost.astype(np.int64)
    s, d = inst.supply.astype(np.int64).tolist(), inst.demand.astype(np.int64).tolist()
    flow, i, j = {}, 0, 0
    while len(flow) < m + n - 1:
        q = min(s[i], d[j])
        flow[(i, j)] = q
        s[i] -= q
        d[j] -= q
        if (s[i] == 0 and i < m - 1) or j == n - 1:
            i += 1
        else:
            j += 1
    for _ in range(limit):
        near = [[] for _ in range(m + n)]
        for a, b in flow:
            near[a].append(m + b)
            near[m + b].append(a)
        dual, up, todo = np.zeros(m + n, np.int64), {0: None}, [0]
        for x in todo:
            for y in near[x]:
                if y not in up:
                    up[y] = x
                    a, b = min(x, y), max(x, y) - m
                    dual[y] = cost[a, b] - dual[x]
                    todo.append(y)
        red = cost - dual[:m, None] - dual[None, m:]
        e = int(np.argmin(red))
        if red.flat[e] >= 0:
            return sum(q * int(cost[c]) for c, q in flow.items())

        def root_path(x):
            path = [x]
            while up[path[-1]] is not None:
                path.append(up[path[-1]])
            return path

        a, b = divmod(e, n)
        left, right = root_path(m + b), root_path(a)
        while len(left) > 1 and len(right) > 1 and left[-2] == right[-2]:
            left.pop()
            right.pop()
        loop = left + right[-2::-1]  # column b .. apex .. row a
        arcs = [(min(x, y), max(x, y) - m) for x, y in zip(loop, loop[1:])]
        out = min(arcs[0::2], key=lambda c: flow[c])
        q = flow[out]
        for k, c in enumerate(arcs):
            flow[c] += q if k % 2 else -q
        del flow[out]
        flow[(a, b)] = q
    return None


def exact(case, seed):
    """The objective of single solves of up to 20000 cells; larger ones take too long here."""
    if "m" not in case or case["m"] * case["n"] > 20000:
        return None
    best = _optimum(_instances(case, seed)[0])
    if best is None:
        return None
    rest = ("iterations", "rows", "cols", "flows", "u", "v") if case["pricing"] == "dantzig" else ("plan",)
    return dict(objective=best, status=0, **{k: None for k in rest})

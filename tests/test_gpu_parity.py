"""GPU parity: the HIP engine against the CPU oracle, through the C ABI.

Bar: bit-exact.  With Dantzig pricing the device follows the sequential reference's
rules, so objective, pivot count, the basis slot by slot and the duals must all equal
the oracle's.  With the faster pricing rules the pivot sequence differs; the int64
objective must still equal the oracle's and every basis must pass the LP optimality
certificate (exact primal sums, an (m+n-1)-arc spanning tree, all reduced costs >= 0).
"""
import json
import os
import sys

import numpy as np
import pytest

import flock_amd as F
import oracle
from flock_amd import instances as I

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden")
EXPECTED = json.load(open(os.path.join(GOLD, "expected.json")))
GPU_OK = {k: v for k, v in EXPECTED.items()}


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def certify(inst, s):
    bad, obj = oracle.certify(inst.cost, inst.supply, inst.demand, s.rows, s.cols, s.flows.astype(np.int64),
                              s.u.astype(np.int64), s.v.astype(np.int64))
    return bad, obj


def assert_same_as_oracle(inst, s, o, exact_sequence):
    assert s.status == 0, (s.status, F.last_error())
    assert s.objective == o.objective
    bad, obj = certify(inst, s)
    assert bad == 0 and obj == s.objective
    if exact_sequence:
        assert s.iterations == o.iterations
        assert np.array_equal(s.rows, o.rows) and np.array_equal(s.cols, o.cols)
        assert np.array_equal(s.flows.astype(np.int64), o.flows)
        assert np.array_equal(s.u.astype(np.int64), o.u) and np.array_equal(s.v.astype(np.int64), o.v)
        assert s.n_flows == o.nonzero_flows


def fits_int32_engine(inst):
    return (2 * (inst.m + inst.n) + 1) * int(inst.cost.max()) < 2 ** 31 - 1


@pytest.mark.parametrize("name", sorted(EXPECTED))
def test_golden_fixtures_dantzig(name):
    from conftest import load_golden
    inst = load_golden(name)
    say("golden", name, inst.m, inst.n)
    if not fits_int32_engine(inst):
        with pytest.raises(F.FlockError) as ei:
            F.solve(inst)
        assert ei.value.status == F.E_RANGE
        return
    s = F.solve(inst, pricing="dantzig")
    o = oracle.solve(inst.cost, inst.supply, inst.demand)
    assert s.objective == EXPECTED[name]["optimum"]
    assert_same_as_oracle(inst, s, o, exact_sequence=True)


def _rand(rng, m, n, cmax=50, smax=100, zeros=False):
    cost = rng.integers(1, cmax + 1, size=(m, n)).astype(np.int32)
    supply = rng.integers(0 if zeros else 1, smax + 1, size=m).astype(np.int32)
    supply[0] += 1
    if zeros:
        cuts = np.sort(rng.integers(0, int(supply.sum()) + 1, size=n - 1))
        demand = np.diff(np.concatenate([[0], cuts, [supply.sum()]])).astype(np.int32)
    else:
        demand = I.balance_demands(rng, supply, 1, smax, n) if supply.sum() >= n else None
        if demand is None:
            return _rand(rng, m, n, cmax, smax, zeros=True)
    return I.Instance(cost, supply, demand)


SHAPES = [(1, 1), (1, 7), (7, 1), (2, 2), (3, 5), (16, 16), (17, 33), (64, 3), (3, 64), (100, 100),
          (128, 257), (300, 40), (511, 512)]


@pytest.mark.parametrize("shape", SHAPES)
def test_random_shapes_dantzig_exact_sequence(shape):
    rng = np.random.default_rng(1000 + shape[0] * 7 + shape[1])
    for zeros in (False, True):
        inst = _rand(rng, *shape, zeros=zeros)
        say("shape", shape, "zeros", zeros)
        s = F.solve(inst, pricing="dantzig")
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        assert_same_as_oracle(inst, s, o, exact_sequence=True)


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_plain_100x100_dantzig(seed):
    inst = I.plain_small(seed)
    say("plain100 seed", seed)
    s = F.solve(inst, pricing="dantzig")
    o = oracle.solve(inst.cost, inst.supply, inst.demand)
    assert_same_as_oracle(inst, s, o, exact_sequence=True)


@pytest.mark.parametrize("pricing", ["candidates", "multi"])
def test_fast_pricing_objective_and_certificate(pricing):
    rng = np.random.default_rng(77)
    for shape in [(5, 9), (40, 60), (100, 100), (257, 130)]:
        inst = _rand(rng, *shape)
        say("pricing", pricing, shape)
        s = F.solve(inst, pricing=pricing)
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        assert_same_as_oracle(inst, s, o, exact_sequence=False)


@pytest.mark.parametrize("cost,supply,demand", [
    ([[2, 2], [6, 4], [5, 8]], [5, 7, 2], [6, 8]),          # argmax tie: the last maximum wins
    ([[8, 1, 9], [2, 2, 4]], [6, 4], [6, 1, 3]),            # stale penalties of the other kind
])
def test_vogel_tie_and_stale_rules_on_device(cost, supply, demand):
    """The two hand-derived Vogel pins of the oracle tests: the device's initial basis
    (one pivot budget: the same basis must come out) and full solve equal the oracle's."""
    inst = I.Instance(np.array(cost, np.int32), np.array(supply, np.int32), np.array(demand, np.int32))
    r, c, f = oracle.vogel(inst.cost, inst.supply, inst.demand)
    for threads in (64, 256):
        s = F.solve(inst, pricing="dantzig", max_iterations=1, threads=threads, team=1 if threads == 64 else 0)
        o = oracle.solve(inst.cost, inst.supply, inst.demand, max_iterations=1)
        assert np.array_equal(s.rows, o.rows) and np.array_equal(s.flows.astype(np.int64), o.flows)
        s = F.solve(inst, pricing="dantzig", threads=threads, team=1 if threads == 64 else 0)
        assert_same_as_oracle(inst, s, oracle.solve(inst.cost, inst.supply, inst.demand), exact_sequence=True)
    assert len(r) == inst.m + inst.n - 1 and int(f.sum()) == int(inst.supply.sum())


def test_nwc_initial_matches_oracle():
    for seed in (4, 5):
        inst = I.plain_small(seed)
        say("nwc seed", seed)
        s = F.solve(inst, pricing="dantzig", initial="nwc")
        o = oracle.solve(inst.cost, inst.supply, inst.demand, initial="nwc")
        assert_same_as_oracle(inst, s, o, exact_sequence=True)


def test_degenerate_family_small_exact():
    inst = I.degenerate(seed=3, m=200, n=100)
    say("degenerate 200x100")
    s = F.solve(inst, pricing="dantzig")
    o = oracle.solve(inst.cost, inst.supply, inst.demand)
    assert_same_as_oracle(inst, s, o, exact_sequence=True)


def test_iteration_budget_reported():
    inst = I.plain_small(1)
    s = F.solve(inst, pricing="dantzig", max_iterations=5)
    assert s.status == F.E_ITERATION_LIMIT and s.iterations == 5
    o = oracle.solve(inst.cost, inst.supply, inst.demand, max_iterations=5)
    # the budget stops both at the same basis
    assert np.array_equal(s.rows, o.rows) and np.array_equal(s.flows.astype(np.int64), o.flows)


def test_batch_equals_plain_solves():
    insts = I.batch(seed=5, count=48)
    say("batch 48")
    sols, ms = F.batch_solve(insts, pricing="dantzig")
    assert ms > 0
    for inst, s in zip(insts, sols):
        p = F.solve(inst, pricing="dantzig")
        assert s.status == 0 and s.objective == p.objective and s.iterations == p.iterations
        assert np.array_equal(s.rows, p.rows) and np.array_equal(s.flows, p.flows)
        assert certify(inst, s)[0] == 0


@pytest.mark.parametrize("threads,team", [(64, 1), (64, 2), (64, 4), (256, 0), (512, 0), (1024, 0)])
def test_every_kernel_configuration_exact(threads, team):
    """Wavefront-per-instance (1, 2 or 4 per workgroup) and workgroup-per-instance
    engines all follow the same pivot sequence as the oracle."""
    rng = np.random.default_rng(31 + threads + team)
    for shape in [(5, 9), (37, 61), (120, 130)]:
        inst = _rand(rng, *shape)
        say("cfg", threads, team, shape)
        s = F.solve(inst, pricing="dantzig", threads=threads, team=team)
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        assert_same_as_oracle(inst, s, o, exact_sequence=True)
        for pricing in ("candidates", "multi"):
            c = F.solve(inst, pricing=pricing, threads=threads, team=team)
            assert c.objective == o.objective and certify(inst, c)[0] == 0, pricing


# (m, n) at the edges of a sweep block of kSlots * threads vectors (2048 at 256 threads,
# 256 for a wavefront): one vector per row with one block, one row more or less; whole
# blocks; a last block of one row; rows longer than a wavefront's block
SWEEP_EDGES = {64: [(255, 3), (257, 4), (63, 16), (65, 16), (3, 1024), (4, 1025), (2, 1540)],
               256: [(2047, 4), (2049, 3), (255, 32), (257, 30), (512, 32), (31, 260), (32, 258), (63, 260)],
               512: [(511, 32), (513, 31), (62, 260), (63, 257)],
               1024: [(1023, 32), (1025, 29), (127, 257)]}


@pytest.mark.parametrize("threads", sorted(SWEEP_EDGES))
def test_sweep_block_edges_exact(threads):
    """The sweep's argmin and ties at block edges: the whole Dantzig sequence equals the
    oracle's (integers, no tolerance); candidate pricing reaches the same objective."""
    rng = np.random.default_rng(77 + threads)
    for k, (m, n) in enumerate(SWEEP_EDGES[threads]):
        inst = _rand(rng, m, n, cmax=(3, 50, 9000)[k % 3], zeros=n > 20 * m)
        say("sweep edge", threads, m, n)
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        assert_same_as_oracle(inst, F.solve(inst, pricing="dantzig", threads=threads), o, exact_sequence=True)
        c = F.solve(inst, pricing="candidates", threads=threads)
        assert c.objective == o.objective and certify(inst, c)[0] == 0


@pytest.mark.parametrize("sizes", [[(1, 1)], [(1, 2), (3, 5), (2, 1)], [(17, 33), (1500, 1500), (5, 6), (64, 63)],
                                   [(600, 701)] * 7 + [(9, 250)]])
def test_batch_packed_copies(sizes):
    """A batch's packed upload (pieces of 8 MiB, one instance larger than a piece, a piece
    that ends between instances, padded and unpadded rows) and its one download: every
    result certified, its arrays the instance's own, objectives equal to plain solves."""
    rng = np.random.default_rng(len(sizes))
    insts = [_rand(rng, m, n, cmax=900) for m, n in sizes]
    say("packed batch", sizes)
    b = F.Batch(insts)
    b.run(pricing="candidates")
    full, short = b.results(), b.results(full=False)
    b.close()
    for inst, s, q in zip(insts, full, short):
        p = F.solve(inst, pricing="candidates")
        assert s.status == 0 and s.objective == q.objective == p.objective
        assert s.iterations == q.iterations and s.n_flows == q.n_flows == len(s.flow_list)
        assert certify(inst, s) == (0, s.objective)
        pos = s.flows != 0
        assert np.array_equal(s.flow_list, np.stack([s.rows[pos], s.cols[pos], s.flows[pos]], axis=1))


def test_batch_results_for_some_instances_and_from_threads():
    """Arrays only where a result asks for them (runs of askers at both ends and alone), and
    one batch's results read by several threads at a time."""
    import threading
    rng = np.random.default_rng(77)
    insts = [_rand(rng, int(m), int(n), cmax=300) for m, n in rng.integers(1, 60, size=(40, 2))]
    say("some results")
    b = F.Batch(insts)
    b.run(pricing="dantzig")
    whole = b.results()
    ask = {0, 1, 5, 17, 18, 19, 39}
    res = (F._Result * len(insts))()
    keep = {}
    for k in ask:
        res[k], keep[k] = F._result_buffers(insts[k].m, insts[k].n)
    assert F.lib().flock_batch_results(b._h, res) == 0
    for k, w in enumerate(whole):
        assert res[k].objective == w.objective and res[k].n_flows == w.n_flows
        if k in ask:
            s = F._solution(res[k], keep[k])
            for f in ("rows", "cols", "flows", "u", "v", "flow_list"):
                assert np.array_equal(getattr(s, f), getattr(w, f)), (k, f)
    got = [None] * 8

    def read(i):
        got[i] = [b.results() for _ in range(5)]
    ts = [threading.Thread(target=read, args=(i,)) for i in range(len(got))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for runs in got:
        for sols in runs:
            for s, w in zip(sols, whole):
                assert s.objective == w.objective
                for f in ("rows", "cols", "flows", "u", "v", "flow_list"):
                    assert np.array_equal(getattr(s, f), getattr(w, f))
    b.close()


# Vogel's register mode: m+n at the edges of 4 and 8 lines per rank, with few distinct costs
# (one covered line lists many others) and with many
VOGEL_EDGES = [(64, 100, 156), (64, 100, 157), (256, 23, 1000), (256, 24, 1000), (256, 1000, 25), (512, 48, 2000),
               (512, 49, 2000), (512, 96, 4000), (512, 97, 4000), (0, 170, 1878), (0, 130, 3966), (0, 130, 3967)]


@pytest.mark.parametrize("threads,m,n", VOGEL_EDGES)
@pytest.mark.parametrize("cmax", [3, 20000])
def test_vogel_line_slots_exact(threads, m, n, cmax):
    """The initial basis, slot by slot (after one Dantzig pivot on both sides), equals the
    oracle's: integers, no tolerance."""
    rng = np.random.default_rng(m + n + cmax)
    inst = _rand(rng, m, n, cmax=cmax, smax=900, zeros=cmax == 3)
    say("vogel edge", threads, m, n, cmax)
    s = F.solve(inst, pricing="dantzig", threads=threads, max_iterations=1)
    o = oracle.solve(inst.cost, inst.supply, inst.demand, max_iterations=1)
    assert s.iterations == o.iterations
    assert np.array_equal(s.rows, o.rows) and np.array_equal(s.cols, o.cols)
    assert np.array_equal(s.flows.astype(np.int64), o.flows)
    assert np.array_equal(s.u.astype(np.int64), o.u) and np.array_equal(s.v.astype(np.int64), o.v)


# deep trees: a north-west corner start's has about 0.66 (m+n) levels when m = n, one or two
# at m = 1 or n = 1; scratch in LDS, in global memory, and with the tree in global memory
@pytest.mark.parametrize("threads,m,n", [(0, 1, 1), (0, 1, 40), (0, 40, 1), (64, 90, 91), (256, 300, 299), (512, 700, 701),
                                         (1024, 2100, 2050), (0, 2000, 2001), (0, 4100, 4001)])
def test_northwest_corner_tree_exact(threads, m, n):
    """The tree of a north-west corner start: basis, duals and flows after one Dantzig pivot
    equal the oracle's."""
    rng = np.random.default_rng(m * 7 + n)
    inst = _rand(rng, m, n, cmax=60, smax=900)
    say("nwc tree", threads, m, n)
    s = F.solve(inst, pricing="dantzig", initial="nwc", threads=threads, max_iterations=1)
    o = oracle.solve(inst.cost, inst.supply, inst.demand, initial="nwc", max_iterations=1)
    assert s.iterations == o.iterations
    assert np.array_equal(s.rows, o.rows) and np.array_equal(s.cols, o.cols)
    assert np.array_equal(s.flows.astype(np.int64), o.flows)
    assert np.array_equal(s.u.astype(np.int64), o.u) and np.array_equal(s.v.astype(np.int64), o.v)


def test_batch_mixed_configurations():
    """One batch mixing wavefront and workgroup classes, candidates pricing."""
    rng = np.random.default_rng(8)
    insts = [_rand(rng, int(a), int(b)) for a, b in [(20, 30), (700, 300), (64, 64), (1500, 900), (3, 400)]]
    say("mixed batch")
    sols, _ = F.batch_solve(insts, pricing="candidates")
    for inst, s in zip(insts, sols):
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        assert s.status == 0 and s.objective == o.objective and certify(inst, s)[0] == 0




def _random_batch(seed, count):
    """Seeded mixed instances: m, n log-uniform in [1, 200], cost ranges from 1 (ties
    everywhere) to 10^4, zero supplies in a third of them (and zero demands where the
    random cuts meet), n often not a multiple of 4."""
    rng = np.random.default_rng(seed)
    sizes = I.log_uniform_sizes(rng, 2 * count, 1, 200)
    out = []
    for k in range(count):
        m, n = int(sizes[2 * k]), int(sizes[2 * k + 1])
        cmax = int(rng.choice([1, 5, 100, 10_000]))
        cost = rng.integers(1, cmax + 1, size=(m, n)).astype(np.int32)
        supply = rng.integers(1, 1001, size=m).astype(np.int32)
        if k % 3 == 0:
            supply[rng.random(m) < 0.3] = 0
        supply[0] += 1
        cuts = np.sort(rng.integers(0, int(supply.sum()) + 1, size=n - 1))
        demand = np.diff(np.concatenate([[0], cuts, [supply.sum()]])).astype(np.int32)
        out.append(I.Instance(cost, supply, demand))
    return out


@pytest.mark.parametrize("threads", [0, 64, 1024])
def test_random_batch_dantzig_exact(threads):
    """256 seeded instances in one batch launch (the default size-class policy, or every
    instance on one-wavefront groups, or on 1024-thread workgroups):
    every one follows the oracle pivot for pivot -- objective, pivot count, basis slot by
    slot, flows and duals."""
    insts = _random_batch(900 + threads, 256)
    say("random batch of", len(insts), "threads", threads)
    b = F.Batch(insts)
    try:
        b.run("dantzig", threads=threads)
        sols = b.results()
    finally:
        b.close()
    for k, (inst, s) in enumerate(zip(insts, sols)):
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        try:
            assert_same_as_oracle(inst, s, o, exact_sequence=True)
        except AssertionError:
            say("instance", k, inst.m, inst.n)
            raise


@pytest.mark.parametrize("pricing", ["candidates", "multi", "switch"])
def test_random_batch_fast_pricing_certified(pricing):
    """The same kind of batch under the faster pricing rules: every objective equals the
    oracle's and every basis passes the exact certificate."""
    insts = _random_batch(1300, 256)
    say("random batch of", len(insts), "pricing", pricing)
    sols, _ = F.batch_solve(insts, pricing=pricing)
    for k, (inst, s) in enumerate(zip(insts, sols)):
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        bad, obj = certify(inst, s)
        assert s.status == 0 and s.objective == o.objective and bad == 0 and obj == s.objective, (k, inst.m, inst.n)

def _edge_instances():
    """Instances at the edges of the int32 range contract ((2(m+n)+1) * max cost < 2^31,
    total supply < 2^31): the largest costs it admits, costs of 0 beside them, one cost
    everywhere (every basis optimal, ties throughout), and a total supply of 2^31 - 1."""
    rng = np.random.default_rng(4242)
    m, n = 37, 53  # n is not a multiple of 4: every row has padding cells
    cmax = (2 ** 31 - 2) // (2 * (m + n) + 1)
    supply = rng.integers(1, 1_000_001, size=m).astype(np.int32)
    demand = I.balance_demands(rng, supply, 1, 1_000_000, n)
    top = rng.integers(cmax // 2, cmax + 1, size=(m, n)).astype(np.int32)
    top[0, 0] = cmax
    zero_top = np.where(rng.random((m, n)) < 0.5, 0, cmax).astype(np.int32)
    flat = np.full((m, n), 7, np.int32)
    out = [("largest costs", I.Instance(top, supply, demand)),
           ("costs 0 or largest", I.Instance(zero_top, supply, demand)),
           ("one cost everywhere", I.Instance(flat, supply, demand))]
    big = np.array([715827882, 715827882, 715827883], np.int32)  # sums to 2^31 - 1
    dem = np.array([429496729] * 4 + [429496731], np.int32)
    assert int(big.sum()) == int(dem.sum()) == 2 ** 31 - 1
    c5 = rng.integers(0, (2 ** 31 - 2) // 17 + 1, size=(3, 5)).astype(np.int32)
    out.append(("total supply 2^31 - 1", I.Instance(c5, big, dem)))
    return out


@pytest.mark.parametrize("threads,team", [(64, 1), (256, 0), (1024, 0)])
def test_range_contract_edges_exact(threads, team):
    """At the edges of the range contract every engine follows the oracle's pivot
    sequence with Dantzig pricing (the oracle keeps duals and flows in int64), and the
    candidate rule's basis passes the exact certificate with the oracle's objective."""
    for what, inst in _edge_instances():
        assert (2 * (inst.m + inst.n) + 1) * int(inst.cost.max()) < 2 ** 31 - 1
        say("range edge", what, "threads", threads)
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        s = F.solve(inst, pricing="dantzig", threads=threads, team=team)
        assert_same_as_oracle(inst, s, o, exact_sequence=True)
        c = F.solve(inst, pricing="candidates", threads=threads, team=team)
        assert c.status == 0 and c.objective == o.objective and certify(inst, c)[0] == 0, what
    # one past the contract is refused before any device work
    m, n = 37, 53
    over = np.full((m, n), (2 ** 31 - 2) // (2 * (m + n) + 1) + 1, np.int32)
    sup = np.full(m, n, np.int32)
    with pytest.raises(F.FlockError) as ei:
        F.solve(I.Instance(over, sup, np.full(n, m, np.int32)))
    assert ei.value.status == F.E_RANGE

@pytest.mark.parametrize("threads", [512, 1024])
def test_large_graph_path_1000x1000(threads):
    """1000x1000 runs as a graph of sweep-grid and pivot-round kernels (set-up and round
    workgroups of 512 or 1024 threads): Dantzig equals the oracle pivot for pivot; the
    candidate, multi-pivot and switch rules reach the same certified optimum."""
    inst = I.plain_large(2)
    say("graph path 1000x1000, threads", threads)
    assert inst.m * inst.n >= F.get_tuning()["graph_min_cells"] > 0
    before = F.get_tuning()
    try:
        F.set_tuning(large_threads=threads)
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        s = F.solve(inst, pricing="dantzig")
        assert_same_as_oracle(inst, s, o, exact_sequence=True)
        assert s.sweeps == s.iterations + 1
        for pricing in ("candidates", "multi", "switch"):
            c = F.solve(inst, pricing=pricing)
            assert c.status == 0 and c.objective == o.objective and certify(inst, c)[0] == 0, pricing
    finally:
        F.set_tuning(**before)



def test_large_graph_path_range_contract_edges():
    """The graph path at the edges of the range contract: 500x502 (padding cells in every
    row) with costs up to the largest it admits -- Dantzig equals the oracle pivot for
    pivot, candidates reach its optimum with a certified basis -- and with one cost
    everywhere (Vogel's basis is already optimal: no pivot)."""
    rng = np.random.default_rng(4343)
    m, n = 500, 502
    cmax = (2 ** 31 - 2) // (2 * (m + n) + 1)
    supply = rng.integers(1, 100_001, size=m).astype(np.int32)
    demand = I.balance_demands(rng, supply, 1, 100_000, n)
    top = rng.integers(cmax // 2, cmax + 1, size=(m, n)).astype(np.int32)
    top[m - 1, n - 1] = cmax
    assert m * n >= F.get_tuning()["graph_min_cells"] > 0
    inst = I.Instance(top, supply, demand)
    say("graph path, largest costs 500x502")
    o = oracle.solve(inst.cost, inst.supply, inst.demand)
    s = F.solve(inst, pricing="dantzig")
    assert_same_as_oracle(inst, s, o, exact_sequence=True)
    c = F.solve(inst, pricing="candidates")
    assert c.status == 0 and c.objective == o.objective and certify(inst, c)[0] == 0
    flat = I.Instance(np.full((m, n), 3, np.int32), supply, demand)
    say("graph path, one cost everywhere 500x502")
    o = oracle.solve(flat.cost, flat.supply, flat.demand)
    for pricing in ("dantzig", "candidates"):
        f = F.solve(flat, pricing=pricing)
        assert f.iterations == 0 and o.iterations == 0
        assert f.status == 0 and f.objective == o.objective == 3 * int(supply.sum())
        assert certify(flat, f)[0] == 0

def test_large_graph_path_degenerate_4000x2000():
    """The degenerate 4000x2000 family (costs in 1..8, ties everywhere) through the graph
    path: certified optimal (exact primal sums, spanning tree, reduced costs >= 0)."""
    inst = I.degenerate(seed=1)
    say("graph path degenerate 4000x2000")
    for pricing in ("candidates", "dantzig", "multi"):
        s = F.solve(inst, pricing=pricing)
        assert s.status == 0, (pricing, s.status, F.last_error())
        bad, obj = certify(inst, s)
        assert bad == 0 and obj == s.objective


def test_large_path_vogel_eight_lines_per_rank():
    """m+n between 4096 and 8192 on the large-instance path: Vogel's set-up kernel keeps
    8 lines per rank in registers, with the tracked keys in global scratch (they do not
    fit LDS beside the line state).  Stopped after one Dantzig pivot, the basis, flows
    and duals equal the oracle's (status 1: the iteration budget)."""
    inst = I.random_instance(np.random.default_rng(4200), 600, 3600, 1000, 10000)
    say("large path, Vogel 8 lines per rank, 600x3600")
    o = oracle.solve(inst.cost, inst.supply, inst.demand, max_iterations=1)
    s = F.solve(inst, pricing="dantzig", max_iterations=1)
    assert o.status == 1 and s.status == 1 and s.iterations == o.iterations == 1
    assert np.array_equal(s.rows, o.rows) and np.array_equal(s.cols, o.cols)
    assert np.array_equal(s.flows.astype(np.int64), o.flows)
    assert np.array_equal(s.u.astype(np.int64), o.u) and np.array_equal(s.v.astype(np.int64), o.v)


@pytest.mark.parametrize("shape", [(20, 8200), (8100, 6)])
def test_tree_beyond_lds_exact(shape):
    """m+n above 8000: the basis tree no longer fits one workgroup's LDS, so flock_solve
    takes the large-instance path with the tree kept in global memory (Vogel's line state
    too when it does not fit).  Dantzig equals the oracle pivot for pivot; the other
    rules reach the same certified optimum."""
    rng = np.random.default_rng(shape[0] + 7 * shape[1])
    inst = I.random_instance(rng, *shape, 1000, 10000)
    say("tree beyond LDS", shape)
    o = oracle.solve(inst.cost, inst.supply, inst.demand)
    s = F.solve(inst, pricing="dantzig")
    assert_same_as_oracle(inst, s, o, exact_sequence=True)
    for pricing in ("candidates", "multi", "switch"):
        c = F.solve(inst, pricing=pricing)
        assert c.status == 0 and c.objective == o.objective and certify(inst, c)[0] == 0, pricing


def test_reference_largest_shape_1000x10000():
    """The reference's largest logged instance shape (1000 x 10000, results/parallel_uv:1423),
    with costs U{1..1000} and supplies/demands U{1..10000}: certified optimal with the
    candidate and switch rules, and both reach the same objective."""
    inst = I.random_instance(np.random.default_rng(10000), 1000, 10000, 1000, 10000)
    say("1000x10000")
    a = F.solve(inst, pricing="candidates")
    assert a.status == 0 and certify(inst, a)[0] == 0
    b = F.solve(inst, pricing="switch")
    assert b.status == 0 and certify(inst, b)[0] == 0 and b.objective == a.objective


def test_instances_too_large_for_256_thread_lds_use_the_1024_engine():
    """A 256- or 512-thread engine needs the tree and the pivot snapshot in LDS; larger
    instances asked for with those sizes (explicitly, or by a size policy) are solved by
    the 1024-thread engine: certified optimal, same objective as the graph path."""
    big = I.degenerate(seed=2, m=2400, n=1600)
    small = I.plain_small(3)
    say("routing 2400x1600 with threads=256")
    ref = F.solve(big, pricing="candidates")
    assert ref.status == 0
    for threads in (256, 512):
        s = F.solve(big, pricing="candidates", threads=threads)
        assert s.status == 0, (threads, s.status, F.last_error())
        bad, obj = certify(big, s)
        assert bad == 0 and obj == s.objective == ref.objective
    before = F.get_tuning()
    try:
        F.set_tuning(wg256_max_v=8000)
        sols, _ = F.batch_solve([big, small, big], pricing="candidates")
        assert [x.status for x in sols] == [0, 0, 0]
        assert sols[0].objective == sols[2].objective == ref.objective
        o = oracle.solve(small.cost, small.supply, small.demand)
        assert sols[1].objective == o.objective
    finally:
        F.set_tuning(**before)


@pytest.mark.parametrize("m,n", [(707, 707), (708, 707), (2500, 200), (131, 3590)])
def test_candidates_on_both_sides_of_the_graph_threshold(m, n):
    """Just under and over 500 000 cells, and an instance whose snapshot does not fit the
    512-thread engine's LDS (graph path from 250 000 cells): the oracle's optimum, certified."""
    inst = I.random_instance(np.random.default_rng(m + n), m, n, 1000, 100 * max(m, n))
    say("graph threshold", m, n)
    s = F.solve(inst, pricing="candidates")
    assert s.status == 0 and certify(inst, s) == (0, s.objective)
    assert s.objective == oracle.solve(inst.cost, inst.supply, inst.demand).objective


def test_autotune_installs_a_policy_with_identical_objectives():
    """flock_autotune measures policies on a sample, requires identical objectives from
    every one (it fails otherwise), and installs the fastest."""
    insts = I.batch(seed=9, count=96)
    before = F.get_tuning()
    say("autotune 96")
    try:
        tuning, ms = F.autotune(insts, pricing="candidates")
        assert ms > 0 and F.get_tuning() == tuning
        sols, _ = F.batch_solve(insts, pricing="candidates")
        for inst, s in zip(insts[:20], sols[:20]):
            o = oracle.solve(inst.cost, inst.supply, inst.demand)
            assert s.status == 0 and s.objective == o.objective
    finally:
        F.set_tuning(**before)


@pytest.mark.parametrize("pricing,count,lo,hi", [("dantzig", 40, 20, 120), ("candidates", 40, 20, 120),
                                                 ("dantzig", 300, 60, 215)])
def test_autotune_keeps_thresholds_the_sample_does_not_depend_on(pricing, count, lo, hi):
    """A batch of at most one instance per compute unit, and a Dantzig batch that takes 512
    threads for its largest instances, launch the same whatever wg256_max_v is."""
    rng = np.random.default_rng(count + hi)
    insts = [_rand(rng, int(m), int(n), cmax=500, smax=900) for m, n in rng.integers(lo, hi + 1, size=(count, 2))]
    before = F.get_tuning()
    say("autotune thresholds", pricing, count)
    try:
        tuning, _ = F.autotune(insts, pricing=pricing)
        assert tuning["wg256_max_v"] == before["wg256_max_v"]
    finally:
        F.set_tuning(**before)


def test_autotune_large_picks_a_tile_shape_with_the_same_optimum():
    """flock_autotune_large tries every sweep tile shape on one large instance, requires the
    same objective from each (it fails otherwise) and installs the fastest; the installed
    shape solves to the oracle's optimum, and Dantzig stays pivot for pivot the oracle's
    whatever the shape."""
    inst = I.random_instance(np.random.default_rng(77), 600, 500, 1000, 10000)
    before = F.get_tuning()
    say("autotune_large 600x500")
    try:
        tuning, ms = F.autotune_large(inst, pricing="candidates")
        assert ms > 0 and tuning["sweep_vectors"] in (1, 2, 4, 8) and tuning["large_threads"] in (512, 1024)
        assert F.get_tuning() == tuning
        o = oracle.solve(inst.cost, inst.supply, inst.demand)
        s = F.solve(inst, pricing="candidates")
        assert s.status == 0 and s.objective == o.objective and certify(inst, s)[0] == 0
        for v in (1, 8):
            F.set_tuning(sweep_vectors=v)
            assert_same_as_oracle(inst, F.solve(inst, pricing="dantzig"), o, exact_sequence=True)
    finally:
        F.set_tuning(**before)

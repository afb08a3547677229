"""The workgroup fixpoint's work split, at its edges (needs an MI355X).

A wave revises 64 / Wp arcs of one changed variable at a time (Wp = words per
domain rounded up to a power of two), numbers the units of 64 variables at a
time, and switches from the source's rows to the target's own rows part-way.
The sizes sit on both sides of each of these limits: 63 to 65 and 130
variables, degrees below, at and above 64 / Wp, domains of 1 to 16 words with
full and nearly empty last words, loose and tight relations, tables in between.
All results are exact: domains, outcomes and node sequences equal the oracle's.
"""
import numpy as np
import pytest

import oracle
from cpim_amd import GModelAdapter, GModelOptions, Server, workload
from cpim_amd.model import domains_to_sets, from_tuples

pytestmark = pytest.mark.gpu

# n, d, e, tightness
SHAPES = [
    (2, 1, 1, 0.0), (3, 2, 3, 0.3), (20, 63, 60, 0.86), (63, 64, 300, 0.87), (64, 8, 900, 0.28),
    (65, 33, 70, 0.80), (66, 16, 2145, 0.12), (130, 20, 5000, 0.15), (40, 65, 400, 0.90), (34, 128, 560, 0.93),
    (33, 129, 300, 0.95), (20, 200, 190, 0.96), (18, 257, 150, 0.975), (12, 320, 60, 0.98), (9, 600, 30, 0.992),
    (7, 1024, 20, 0.995),
]


def networks(n, d, e, t, seed):
    return workload.random_binary(n, d, e, t, workload.instance_seed(31, seed), preremove=0.15 if d > 3 else 0.0)


@pytest.mark.parametrize("seed", [0, 1])
@pytest.mark.parametrize("n,d,e,t", SHAPES)
def test_block_fixpoint_equals_oracle(gpu, n, d, e, t, seed):
    desc = networks(n, d, e, t, seed)
    ok, dom, _ = oracle.Oracle(desc).root_ac()
    with GModelAdapter.Build(desc) as m:
        st = m.EnforceGAC_Block()
        assert st.inconsistent == (not ok)
        if not ok:
            return
        assert (m.ReadDomains(0) == dom).all()
        # one more value gone from one variable: propagation from its arcs alone
        v = n // 2
        vals = domains_to_sets(dom, desc.dom_size)[v]
        cut = dom.copy()
        cut[v, vals[0] // 64] &= ~np.uint64(1 << (vals[0] % 64))
        m.WriteDomains(0, cut)
        st = m.EnforceGAC_Block(v)
        ok2, dom2, _ = oracle.Oracle(desc.with_init_dom(cut)).root_ac()
        assert st.inconsistent == (not ok2)
        if ok2:
            assert (m.ReadDomains(0) == dom2).all()


@pytest.mark.parametrize("n,d,e,t", SHAPES)
def test_workgroup_singleton_tests_equal_oracle(gpu, n, d, e, t):
    desc = networks(n, d, e, t, 2)
    o = oracle.Oracle(desc)
    ok, dom, _ = o.root_ac()
    if not ok:
        pytest.skip("the root is inconsistent")
    tests = np.array([(v, a) for v, vals in enumerate(domains_to_sets(dom, desc.dom_size)) for a in vals], np.int32)
    tests = tests[np.linspace(0, len(tests) - 1, min(len(tests), 200)).astype(int)]
    want, _ = o.singleton_tests(tests)
    with GModelAdapter.Build(desc) as m:
        assert not m.EnforceGAC_Block().inconsistent
        got, _ = m.SingletonTests(tests, mode="workgroup")
    assert (got == want).all()


@pytest.mark.parametrize("tables", [0, 3])
@pytest.mark.parametrize("n,d,rho", [(20, 5, 0.5), (64, 10, 0.2), (70, 30, 0.15), (30, 70, 0.3), (25, 140, 0.3)])
def test_search_equals_oracle(gpu, n, d, rho, tables):
    e = int(round(rho * n * (n - 1) / 2))
    base = workload.random_binary(n, d, e, 0.95 * workload.phase_transition_tightness(n, d, rho),
                                  workload.instance_seed(32, n))
    scopes, lists = [list(s) for s in base.scopes()], list(base.tuple_lists())
    rng = np.random.default_rng(n)
    for k in range(tables):  # tables between the binary constraints
        at = int(rng.integers(0, len(scopes) + 1))
        scopes.insert(at, rng.choice(n, 3, replace=False).tolist())
        lists.insert(at, workload.random_table(1000 * n + k, 3, d, min(600, d ** 3 // 2)))
    desc = from_tuples(base.dom_size, scopes, lists)
    want = oracle.Oracle(desc, oracle.AC3 if tables else oracle.AC3BIT).mac(node_limit=300, trace_cap=1000)
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        st, sol, trace = m.Solve(node_limit=300, trace_capacity=1000)
    assert (st.num_solutions, st.num_positive, st.num_negative) == (want.num_sol, want.num_positive, want.num_negative)
    assert trace == want.trace
    if want.num_sol:
        assert (np.asarray(sol) == want.solution).all()


@pytest.mark.parametrize("n,d,e,t", [
    # 1 to 4 arcs a lane at 1024 threads, and past it (4096 arcs); 31 to 33 values
    (80, 2, 500, 0.01), (80, 2, 1030, 0.005), (80, 2, 2047, 0.003), (80, 2, 2049, 0.003),
    (23, 31, 200, 0.30), (23, 32, 200, 0.31), (23, 33, 200, 0.31), (12, 8, 40, 0.45), (3, 1, 3, 0.0),
])
def test_lds_search_equals_oracle(gpu, n, d, e, t):
    desc = workload.random_binary(n, d, e, t, workload.instance_seed(33, n * 100 + d))
    want = oracle.Oracle(desc).mac(node_limit=400, trace_cap=1000)
    with GModelAdapter.Build(desc) as m:
        st, _, trace = m.Solve(node_limit=400, trace_capacity=1000)
    assert (st.num_solutions, st.num_positive, st.num_negative) == (want.num_sol, want.num_positive, want.num_negative)
    assert trace == want.trace


@pytest.mark.parametrize("n,d,e,t,tables", [
    # one and two arcs a lane beside tables, one arc a lane above 16 values;
    # 16 tables and one too many; as many variables as lanes
    (30, 16, 100, 0.35, 4), (30, 16, 240, 0.22, 2), (30, 17, 100, 0.35, 0), (24, 16, 60, 0.35, 16),
    (24, 16, 60, 0.35, 17), (64, 4, 64, 0.3, 1), (65, 4, 64, 0.3, 0), (200, 3, 230, 0.2, 0), (5, 16, 0, 0.0, 2),
])
def test_small_network_searches_equal_oracle(gpu, n, d, e, t, tables):
    """Solve in one go, and on a server in steps of seven nodes (each resumes
    from the stored state)."""
    base = workload.random_binary(n, d, e, t, workload.instance_seed(36, n * 100 + d))
    scopes, lists = [list(s) for s in base.scopes()], list(base.tuple_lists())
    rng = np.random.default_rng(n + d)
    for k in range(tables):  # tables between the binary constraints
        at = int(rng.integers(0, len(scopes) + 1))
        scopes.insert(at, rng.choice(n, 3, replace=False).tolist())
        lists.insert(at, workload.random_table(1000 * n + k, 3, d, min(500, d ** 3 // 2)))
    desc = from_tuples(base.dom_size, scopes, lists)
    want = oracle.Oracle(desc, oracle.AC3 if tables else oracle.AC3BIT).mac(node_limit=300, trace_cap=1000)
    counts = (want.num_sol, want.num_positive, want.num_negative)
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        st, sol, trace = m.Solve(node_limit=300, trace_capacity=1000)
    assert (st.num_solutions, st.num_positive, st.num_negative) == counts
    assert trace == want.trace
    srv = Server(max_slots=1, nodes_per_step=7)
    rid = srv.submit(desc, node_limit=300)
    while not srv.poll():
        srv.step()
    r = srv.result(rid)
    srv.close()
    assert (r["num_positive"], r["num_negative"]) == counts[1:]
    if want.num_sol:
        assert (np.asarray(sol) == want.solution).all() and (np.asarray(r["solution"]) == want.solution).all()


@pytest.mark.parametrize("d,arity,tuples", [
    (16, 3, 512), (16, 3, 513), (17, 3, 512), (16, 4, 500), (16, 5, 300), (15, 3, 449), (8, 4, 448), (9, 2, 40),
    (4, 3, 1), (2, 4, 5), (5, 3, 64), (5, 3, 65), (1, 3, 1),
])
def test_small_tables_equal_oracle(gpu, d, arity, tuples):
    # the one-pass revision of small tables and the forms beyond its limits
    # (16 values, 4 positions, 512 tuples), in every engine that revises tables
    n = 12
    rng = np.random.default_rng(1000 * d + tuples)
    scopes = [rng.choice(n, max(2, arity - (k & 1)), replace=False).tolist() for k in range(7)]
    lists = [workload.random_table(77 * d + k, len(s), d, min(tuples, max(1, d ** len(s) * 3 // 4)))
             for k, s in enumerate(scopes)]
    base = workload.random_binary(n, d, 12, 0.15 if d > 2 else 0.0, workload.instance_seed(34, d))
    desc = from_tuples(base.dom_size, [list(s) for s in base.scopes()] + scopes, list(base.tuple_lists()) + lists)
    o = oracle.Oracle(desc, oracle.AC3)
    ok, dom, _ = o.root_ac()
    want = oracle.Oracle(desc, oracle.AC3).mac(node_limit=200, trace_cap=600)
    opts = GModelOptions(skip_non_binary=False)
    for run in ("EnforceGAC_Block", "EnforceGAC", "EnforceGAC_Persistent"):
        with GModelAdapter.Build(desc, opts) as m:
            st = getattr(m, run)(False) if run != "EnforceGAC_Block" else m.EnforceGAC_Block()
            assert st.inconsistent == (not ok), run
            assert not ok or (m.ReadDomains(0) == dom).all(), run
    with GModelAdapter.Build(desc, opts) as m:
        st, _, trace = m.Solve(node_limit=200, trace_capacity=600)
        assert (st.num_solutions, st.num_positive, st.num_negative) == \
            (want.num_sol, want.num_positive, want.num_negative)
        assert trace == want.trace
    with GModelAdapter.Build(desc, opts) as m:
        sok, sdom, _ = oracle.Oracle(desc, oracle.AC3).sac1()
        st = m.EnforceSAC(mode="workgroup")
        assert st.consistent == sok
        assert not sok or (m.ReadDomains(0) == sdom).all()


@pytest.mark.parametrize("kind", ["binary", "tables", "parallel"])
@pytest.mark.parametrize("n,d,rho", [
    # degrees below and above 64 / Wp constraints, domains of 1 to 5 words
    (25, 6, 0.5), (90, 8, 0.9), (40, 20, 0.3), (25, 70, 0.5), (40, 100, 0.95), (20, 150, 0.5), (24, 300, 0.95),
])
def test_wdeg_search_and_weights_equal_oracle(gpu, n, d, rho, kind):
    # dom/wdeg: fixpoints in AC3's order, many constraints of a variable at a
    # time; tables and parallel constraints take them one after another
    e = int(round(rho * n * (n - 1) / 2))
    desc = workload.random_binary(n, d, e, 0.97 * workload.phase_transition_tightness(n, d, rho),
                                  workload.instance_seed(35, n))
    if kind != "binary":
        scopes, lists = [list(s) for s in desc.scopes()], list(desc.tuple_lists())
        rng = np.random.default_rng(n)
        for k in range(4):
            at = int(rng.integers(0, len(scopes) + 1))
            if kind == "tables":
                scope = rng.choice(n, 3, replace=False).tolist()
                tup = workload.random_table(500 * n + k, 3, d, min(900, d ** 3 // 2))
            else:  # a second constraint on an existing pair, half of them the other way round
                c = int(rng.integers(0, len(scopes)))
                scope, tup = scopes[c][::-1] if k & 1 else scopes[c], lists[c][:, ::-1] if k & 1 else lists[c]
                tup = np.ascontiguousarray(tup[rng.random(len(tup)) < 0.9])
            scopes.insert(at, list(scope))
            lists.insert(at, tup)
        desc = from_tuples(desc.dom_size, scopes, lists)
    algo = oracle.AC3 if kind == "tables" else oracle.AC3BIT
    with oracle.var_heuristic(2):
        o = oracle.Oracle(desc, algo)
        want = o.mac(node_limit=120, trace_cap=600)
        weights = o.weights().copy()
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        st, _, trace = m.Solve(node_limit=120, trace_capacity=600, heuristic="dom/wdeg")
        assert trace == want.trace
        assert (st.num_solutions, st.num_positive, st.num_negative) == \
            (want.num_sol, want.num_positive, want.num_negative)
        assert (m.Weights() == weights).all()


@pytest.mark.parametrize("n,d,e,t", [(60, 37, 500, 0.62), (100, 100, 1650, 0.55), (100, 100, 1690, 0.55)])
def test_sac_pass_same_on_both_sides_of_the_kernel_choice(gpu, n, d, e, t):
    # little work goes to one workgroup per test, more to the bit-sliced
    # kernels (23,068,672 arc words: e = 1673 at n = d = 100)
    desc = workload.random_binary(n, d, e, t, workload.instance_seed(36, e), preremove=0.0)
    with GModelAdapter.Build(desc) as m:
        assert not m.EnforceGAC_Auto().inconsistent
        tests = np.array([(v, a) for v, vals in enumerate(domains_to_sets(m.ReadDomains(0), desc.dom_size))
                          for a in vals], np.int32)
        got = {mode: m.SingletonTests(tests, mode=mode)[0] for mode in ("auto", "sliced", "workgroup")}
    assert (got["auto"] == got["sliced"]).all() and (got["auto"] == got["workgroup"]).all()


GRID_SHAPES = SHAPES + [
    (1030, 1000, 60, 0.993),   # domains above 128 KB: the persistent rounds read them from memory
    (1030, 1000, 40, 0.5),
    (2000, 8, 140000, 0.02),   # more arcs than the persistent grid has lanes
    (300, 250, 4000, 0.96), (300, 130, 4000, 0.93),
]


@pytest.mark.parametrize("mode", ["plain", "persistent"])
@pytest.mark.parametrize("n,d,e,t", GRID_SHAPES)
def test_grid_rounds_equal_oracle(gpu, n, d, e, t, mode):
    # a lane per arc word: tight relations settled by the wave, and a seed of
    # one variable (its constraints in both directions in the first round)
    desc = networks(n, d, e, t, 3)
    ok, dom, _ = oracle.Oracle(desc).root_ac()
    with GModelAdapter.Build(desc) as m:
        run = (lambda v: m.EnforceGAC(False, v)) if mode == "plain" else (lambda v: m.EnforceGAC_Persistent(False, v))
        before = m.ReadDomains(0)
        st = run(-1)
        assert st.inconsistent == (not ok)
        if not ok:
            return
        got = m.ReadDomains(0)
        assert (got == dom).all() and st.converged
        assert st.deletions == int(np.bitwise_count(before).sum()) - int(np.bitwise_count(dom).sum())
        sizes = np.bitwise_count(dom).sum(axis=1)
        for v in range(0, n, max(1, n // 50)):
            assert m.GetDomainSize(v, 0) == sizes[v]
        v = n // 2
        a = int(domains_to_sets(dom, desc.dom_size)[v][0])
        cut = dom.copy()
        cut[v] = 0
        cut[v, a // 64] = np.uint64(1 << (a % 64))
        m.WriteDomains(0, cut)
        st = run(v)
        ok2, dom2, _ = oracle.Oracle(desc.with_init_dom(cut)).root_ac()
        assert st.inconsistent == (not ok2)
        if ok2:
            assert (m.ReadDomains(0) == dom2).all()


@pytest.mark.parametrize("tables", [4, 5, 16, 17, 40])
def test_many_small_tables_equal_oracle(gpu, tables):
    """More tables than the workgroup has waves (4 in a singleton test, 16 in
    the others): a wave takes several, over several rounds."""
    n, d = 24, 16
    base = workload.random_binary(n, d, 60, 0.35, workload.instance_seed(37, 1))
    scopes, lists = [list(s) for s in base.scopes()], list(base.tuple_lists())
    rng = np.random.default_rng(40)
    for k in range(tables):
        at = int(rng.integers(0, len(scopes) + 1))
        scopes.insert(at, rng.choice(n, 3, replace=False).tolist())
        lists.insert(at, workload.random_table(24000 + k, 3, d, 500))
    desc = from_tuples(base.dom_size, scopes, lists)
    o = oracle.Oracle(desc, oracle.AC3)
    want = o.mac(node_limit=300, trace_cap=1000)
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        st, _, trace = m.Solve(node_limit=300, trace_capacity=1000)
        assert (st.num_positive, st.num_negative) == (want.num_positive, want.num_negative)
        assert trace == want.trace
        ok, dom, _ = oracle.Oracle(desc, oracle.AC3).root_ac()
        assert m.EnforceGAC_Block().inconsistent == (not ok)
        if ok:
            assert (m.ReadDomains(0) == dom).all()
            tests = np.array([(v, a) for v, vals in enumerate(domains_to_sets(dom, desc.dom_size)) for a in vals],
                             np.int32)
            got, _ = m.SingletonTests(tests, mode="workgroup")
            assert (got == oracle.Oracle(desc, oracle.AC3).singleton_tests(tests)[0]).all()


@pytest.mark.parametrize("n,d,e,t", [
    # one workgroup up to 800 constraint words, rounds over the grid beyond
    (60, 9, 799, 0.3), (60, 9, 800, 0.3), (60, 9, 801, 0.3), (60, 70, 400, 0.9), (60, 70, 401, 0.9), (150, 20, 5000, 0.1),
])
def test_auto_fixpoint_equals_oracle(gpu, n, d, e, t):
    desc = networks(n, d, e, t, 3)
    ok, dom, _ = oracle.Oracle(desc).root_ac()
    with GModelAdapter.Build(desc) as m:
        assert m.EnforceGAC_Auto().inconsistent == (not ok)
        if not ok:
            return
        assert (m.ReadDomains(0) == dom).all()
        for v in (0, n - 1):  # one variable assigned
            a = domains_to_sets(dom, desc.dom_size)[v][-1]
            cut = dom.copy()
            cut[v] = 0
            cut[v, a // 64] = np.uint64(1 << (a % 64))
            m.WriteDomains(0, cut)
            st = m.EnforceGAC_Auto(v)
            ok2, dom2, _ = oracle.Oracle(desc.with_init_dom(cut)).root_ac()
            assert st.inconsistent == (not ok2)
            if ok2:
                assert (m.ReadDomains(0) == dom2).all()

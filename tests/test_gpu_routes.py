"""Automatic choices between kernels, where the wrong one costs several times
the right one (needs an MI355X)."""
import time

import numpy as np
import pytest

import oracle
from cpim_amd import Batch, GModelAdapter, GModelOptions, workload
from cpim_amd import _native as N
from cpim_amd.model import ModelDesc, domains_to_sets, from_tuples, words_for

pytestmark = pytest.mark.gpu


def with_pairs(pairs, n, d, t, seed=3):
    """Random relations of tightness t over the given pairs of n variables."""
    pairs = np.asarray(pairs, np.int32)
    base = workload.random_binary(max(n, 2 + int(np.sqrt(2 * len(pairs)))), d, len(pairs), t, seed)
    return ModelDesc(np.full(n, d, np.int32), base.con_arity, pairs.reshape(-1), base.bin_rel)


def path(n, d):
    """x0 <= x1 <= ... : a change at one end runs to the other."""
    rel = np.zeros((n - 1, d, words_for(d)), np.uint64)
    for a in range(d):
        for b in range(a, d):
            rel[:, a, b // 64] |= np.uint64(1) << np.uint64(b % 64)
    pairs = np.stack([np.arange(n - 1), np.arange(1, n)], 1).astype(np.int32)
    return ModelDesc(np.full(n, d, np.int32), np.full(n - 1, 2, np.int32), pairs.reshape(-1), rel)


def lattice(k, d, t):
    pairs = [(i * k + j, i * k + j + 1) for i in range(k) for j in range(k - 1)]
    pairs += [(i * k + j, i * k + k + j) for i in range(k - 1) for j in range(k)]
    return with_pairs(pairs, k * k, d, t)


def star(n, d, t):
    return with_pairs([(0, v) for v in range(1, n)], n, d, t)


@pytest.mark.parametrize("name,make,faster", [
    ("path", lambda: path(300, 64), "sliced"),
    ("lattice", lambda: lattice(25, 40, 0.7), "sliced"),
    ("star", lambda: star(600, 16, 0.4), "workgroup"),
    ("dense", lambda: workload.random_binary(60, 37, 500, 0.723, 7), "workgroup"),
])
def test_sac_pass_takes_the_faster_kernel(gpu, name, make, faster):
    desc = make()
    with GModelAdapter.Build(desc) as m:
        assert not m.EnforceGAC_Auto().inconsistent
        tests = np.array([(v, a) for v, vals in enumerate(domains_to_sets(m.ReadDomains(0), desc.dom_size))
                          for a in vals], np.int32)
        fail, ms = {}, {}
        for mode in ("auto", "sliced", "workgroup"):
            for _ in range(3):
                fail[mode], st = m.SingletonTests(tests, mode=mode)
                ms[mode] = min(ms.get(mode, 1e9), st.kernel_ms)
    assert (fail["auto"] == fail["sliced"]).all() and (fail["auto"] == fail["workgroup"]).all()
    slower = "sliced" if faster == "workgroup" else "workgroup"
    # the kernels are 2.5 to 9 times apart: half-way between them, by ratio
    assert ms["auto"] < (ms[faster] * ms[slower]) ** 0.5, ms


@pytest.mark.parametrize("heuristic", ["dom", "dom/wdeg"])
@pytest.mark.parametrize("n,d,e,t", [
    # searches settle tight relations by the wave from 12,288 arc words of
    # three-word domains on: both sides of that line, and wider domains
    (80, 150, 1535, 0.93), (80, 150, 1536, 0.93), (50, 1000, 600, 0.97), (300, 250, 3000, 0.963),
])
def test_tight_search_equals_oracle(gpu, n, d, e, t, heuristic):
    desc = workload.random_binary(n, d, e, t, workload.instance_seed(42, e))
    with oracle.var_heuristic(2 if heuristic == "dom/wdeg" else 0):
        o = oracle.Oracle(desc)
        want = o.mac(node_limit=40, trace_cap=200)
        weights = o.weights().copy()
    with GModelAdapter.Build(desc) as m:
        st, _, trace = m.Solve(node_limit=40, trace_capacity=200, heuristic=heuristic)
        assert (st.num_solutions, st.num_positive, st.num_negative) == \
            (want.num_sol, want.num_positive, want.num_negative)
        assert trace == want.trace
        if heuristic == "dom/wdeg":
            assert (m.Weights() == weights).all()


def test_tight_and_other_units_of_a_batch_equal_oracle(gpu):
    shapes = [(80, 150, 1536, 0.93), (80, 150, 1535, 0.93), (30, 16, 109, 0.4), (25, 140, 90, 0.9), (50, 1000, 600, 0.97)]
    descs = [workload.random_binary(n, d, e, t, workload.instance_seed(43, e + d)) for n, d, e, t in shapes]
    for per_unit in (True, False):
        res, _ = Batch(descs).run(30, persistent=not per_unit)
        for desc, r in zip(descs, res):
            want = oracle.Oracle(desc).mac(node_limit=30)
            assert (r.num_positive, r.num_negative) == (want.num_positive, want.num_negative)


@pytest.mark.parametrize("n,d,e,t", [(300, 250, 20000, 0.963), (300, 250, 3000, 0.963)])
def test_tight_root_of_a_search_takes_no_longer_than_the_fixpoint(gpu, n, d, e, t):
    # the same workgroup fixpoint; without the tight path the search took twice as long
    desc = workload.random_binary(n, d, e, t, 5)
    with GModelAdapter.Build(desc) as m:
        init = m.ReadDomains(0)
        block, root = [], []
        for _ in range(3):
            m.WriteDomains(0, init)
            block.append(m.EnforceGAC_Block().kernel_ms)
            m.WriteDomains(0, init)
            root.append(m.Solve(node_limit=1)[0].gac_time * 1e3)
    assert min(root) < 1.4 * min(block)


@pytest.mark.parametrize("mode", ["plain", "persistent"])
@pytest.mark.parametrize("n,d,e,t", [
    # wide domains on few, tight constraints (a wave takes 16 lanes of arc
    # words), and rounds whose grids differ: the first round of each has fewer
    # workgroups than the later ones
    (60, 1024, 60, 0.995), (100, 1000, 300, 0.99), (300, 250, 4000, 0.96), (500, 250, 20000, 0.963),
    (700, 130, 30000, 0.92),
])
def test_wide_rounds_equal_oracle(gpu, n, d, e, t, mode):
    desc = workload.random_binary(n, d, e, t, 5, preremove=0.1)
    ok, dom, _ = oracle.Oracle(desc).root_ac()
    with GModelAdapter.Build(desc) as m:
        run = (lambda v: m.EnforceGAC(False, v)) if mode == "plain" else (lambda v: m.EnforceGAC_Persistent(False, v))
        st = run(-1)
        assert st.inconsistent == (not ok)
        assert not ok or (m.ReadDomains(0) == dom).all()
        if not ok:
            return
        hit = 0
        for v in (n // 2, n - 1, 0):  # half of one variable's values gone
            cut = dom.copy()
            vals = domains_to_sets(dom, desc.dom_size)[v]
            for a in vals[:(len(vals) + 1) // 2]:
                cut[v, a // 64] &= ~np.uint64(1 << (a % 64))
            m.WriteDomains(0, cut)
            st = run(v)
            ok2, dom2, _ = oracle.Oracle(desc.with_init_dom(cut)).root_ac()
            assert st.inconsistent == (not ok2)
            assert not ok2 or (m.ReadDomains(0) == dom2).all()
            hit += not ok2 or int(np.bitwise_count(dom2).sum()) < int(np.bitwise_count(cut).sum())
        assert hit, "no seed removed anything"


def test_wide_rounds_on_few_constraints_are_not_slower_than_one_workgroup(gpu):
    # one lane per arc word left the rounds of such networks to two workgroups,
    # whose waves settled their arcs one after the other: 785 us, against 297
    # with the arcs spread (and 1070 for the workgroup fixpoint)
    desc = workload.random_binary(60, 1024, 60, 0.995, 5, preremove=0.1)
    with GModelAdapter.Build(desc) as m:
        init = m.ReadDomains(0)
        ms = {}
        for _ in range(3):
            for name, run in (("rounds", lambda: m.EnforceGAC(False)), ("block", m.EnforceGAC_Block)):
                m.WriteDomains(0, init)
                ms[name] = min(ms.get(name, 1e9), run().kernel_ms)
    assert ms["rounds"] < 0.5 * ms["block"], ms


def test_workgroup_rounds_pass_over_unchanged_variables(gpu):
    # one changed variable a round: a round's cost must not grow with the
    # variables that did not change (counting every one, 21 us a round of 3,000
    # variables against 5 us of 700)
    us = {}
    for n in (700, 2800):
        desc = path(n, 64)
        with GModelAdapter.Build(desc) as m:
            cut = m.ReadDomains(0)
            cut[0, 0] = np.uint64(1 << 63)
            for _ in range(3):
                m.WriteDomains(0, cut)
                st = m.EnforceGAC_Block(0)
                assert st.converged and st.deletions == 63 * (n - 1)
                us[n] = min(us.get(n, 1e9), st.kernel_ms * 1e3 / n)
    assert us[2800] < 2.5 * us[700], us


@pytest.mark.parametrize("n,d,seed", [(1000, 64, -1), (1000, 64, 0), (4200, 64, 0)])
def test_auto_does_not_run_a_long_chain_by_rounds_alone(gpu, n, d, seed):
    # a round over the grid costs 8 us however little it does: 7.6 ms against 2.7
    # with the workgroup fixpoint at 1,000, 35 against 23 with the asynchronous
    # kernel at 4,200
    desc = path(n, d)
    with GModelAdapter.Build(desc) as m:
        cut = m.ReadDomains(0)
        cut[0, 0] = np.uint64(1 << (d - 1))
        s = {}
        for _ in range(3):
            for name, run in (("auto", lambda: m.EnforceGAC_Auto(seed)), ("plain", lambda: m.EnforceGAC(False, seed))):
                m.WriteDomains(0, cut)
                t0 = time.perf_counter()
                st = run()
                s[name] = min(s.get(name, 1e9), time.perf_counter() - t0)
                assert st.converged and not st.inconsistent and st.deletions == (d - 1) * (n - 1)
                dom = m.ReadDomains(0)
                assert (dom == np.uint64(1 << (d - 1))).all()
    assert s["auto"] < 0.8 * s["plain"], s


@pytest.mark.parametrize("n,d,wipe", [(900, 8, False), (900, 8, True), (4200, 4, False), (4200, 4, True), (850, 70, False)])
def test_auto_chain_on_an_open_level(gpu, n, d, wipe):
    """The long chain's second kernel answers what the first one's frontier
    does: of variables up to 4,096 constraints, of constraints beyond.  Some
    values are missing along the path; wipe: the chain empties a variable near
    its end."""
    from test_gpu_open_levels import seeded_closure
    desc = path(n, d)
    rng = np.random.default_rng(n + wipe)
    sets = [set(np.flatnonzero(rng.random(d) < 0.7).tolist()) | {0, d - 1} for _ in range(n)]
    sets[0] = {d - 1}
    if wipe:
        sets[n - 10] = set(range(d - 1))
    want = seeded_closure(desc, sets, 0, "constraint" if n - 1 > 4096 else "variable")
    dom = np.zeros((n, words_for(d)), np.uint64)
    for v, s in enumerate(sets):
        for a in s:
            dom[v, a // 64] |= np.uint64(1 << (a % 64))
    with GModelAdapter.Build(desc) as m:
        m.WriteDomains(0, dom)
        st = m.EnforceGAC_Auto(0)
        assert st.inconsistent == (want is None)
        if want is not None:
            assert [set(g) for g in domains_to_sets(m.ReadDomains(0), desc.dom_size)] == want
            assert st.deletions == sum(map(len, sets)) - sum(map(len, want))
        # rounds again, on the control block that the second kernel left
        m.WriteDomains(0, dom)
        ok, full, _ = oracle.Oracle(desc.with_init_dom(dom)).root_ac()
        assert m.EnforceGAC(False).inconsistent == (not ok)
        assert not ok or (m.ReadDomains(0) == full).all()


@pytest.mark.parametrize("n,d", [(2047, 8), (2048, 8), (2049, 8), (4097, 70), (1024, 1), (300, 70), (1638, 300), (9, 1024)])
def test_level_calls_on_many_variables(gpu, n, d):
    # queries by 256 or 1024 threads, levels written in order up to 64 KB through
    # the host box and by copy beyond, the last words of a domain partly used
    rng = np.random.default_rng(n)
    W = words_for(d)
    desc = ModelDesc(np.full(n, d, np.int32), np.full(1, 2, np.int32), np.array([0, n - 1], np.int32),
                     np.full((1, d, W), ~np.uint64(0)))
    dom = rng.integers(0, 1 << 63, (n, W), dtype=np.uint64) | np.uint64(1 << 63) | np.uint64(3)
    cap = np.array([(1 << min(64, max(0, d - 64 * w))) - 1 for w in range(W)], dtype=object)
    want = np.array([[int(x) & c for x, c in zip(row, cap)] for row in dom], dtype=np.uint64)
    sizes = np.bitwise_count(want).sum(axis=1)
    with GModelAdapter.Build(desc) as m:
        m.WriteDomains(0, dom)
        assert (m.ReadDomains(0) == want).all()
        for v in (0, 1, n // 2, n - 1):
            assert m.GetDomainSize(v, 0) == sizes[v]
        open_ = np.flatnonzero(sizes > 1)
        assert m.GetMinDomainVar(0) == (open_[np.argmin(sizes[open_])] if len(open_) else -1)
        assert m.IsFullyAssigned(0) == bool((sizes == 1).all())
        one = np.zeros((n, W), np.uint64)
        one[:, 0] = 1
        m.WriteDomains(0, one)
        assert m.IsFullyAssigned(0) and m.GetMinDomainVar(0) == -1
        if d > 1:
            one[n - 1, 0] = 3
            m.WriteDomains(0, one)
            assert not m.IsFullyAssigned(0) and m.GetMinDomainVar(0) == n - 1


def with_tables(n, d, e, t, tables, arity, tuples):
    base = workload.random_binary(n, d, e, t, 3)
    scopes, lists = [list(s) for s in base.scopes()], list(base.tuple_lists())
    rng = np.random.default_rng(tables)
    for k in range(tables):
        scopes.append(rng.choice(n, arity, replace=False).tolist())
        lists.append(workload.random_table(99 * k + arity, arity, d, tuples))
    return from_tuples(base.dom_size, scopes, lists)


@pytest.mark.parametrize("mode", ["plain", "persistent", "auto", "block"])
@pytest.mark.parametrize("n,d,e,tables,arity,tuples,keep", [
    # one to many tables per wave and workgroup, small and larger ones; values
    # go at the root and after half of one variable's values are gone
    (60, 40, 40, 1, 3, 700, 0.45), (60, 40, 40, 30, 3, 700, 0.45), (150, 40, 100, 300, 3, 800, 0.6),
    (150, 12, 60, 300, 5, 900, 0.62), (100, 16, 40, 300, 3, 400, 0.7), (40, 70, 30, 20, 3, 2500, 0.4),
    (60, 6, 40, 33, 4, 200, 0.7),
])
def test_many_tables_equal_oracle(gpu, n, d, e, tables, arity, tuples, keep, mode):
    desc = with_tables(n, d, e, 0.3, tables, arity, tuples)
    rng = np.random.default_rng(7)
    init = desc.full_domains()
    for v in range(n):  # some values gone, so that tables lose tuples
        for a in range(d):
            if rng.random() > keep and a != v % d:
                init[v, a // 64] &= ~np.uint64(1 << (a % 64))
    desc = desc.with_init_dom(init)
    ok, dom, _ = oracle.Oracle(desc, oracle.AC3).root_ac()
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        run = {"plain": lambda v: m.EnforceGAC(False, v), "persistent": lambda v: m.EnforceGAC_Persistent(False, v),
               "auto": m.EnforceGAC_Auto, "block": m.EnforceGAC_Block}[mode]
        st = run(-1)
        assert st.inconsistent == (not ok)
        if not ok:
            return
        assert (m.ReadDomains(0) == dom).all()
        for v in (int(desc.con_scope[-1]), n // 2):
            vals = domains_to_sets(dom, desc.dom_size)[v]
            cut = dom.copy()
            for a in vals[:len(vals) // 2]:
                cut[v, a // 64] &= ~np.uint64(1 << (a % 64))
            m.WriteDomains(0, cut)
            st = run(v)
            ok2, dom2, _ = oracle.Oracle(desc.with_init_dom(cut), oracle.AC3).root_ac()
            assert st.inconsistent == (not ok2)
            assert not ok2 or (m.ReadDomains(0) == dom2).all()


def test_large_tables_of_a_round_go_to_workgroups_of_their_own(gpu):
    # 30 waves of two workgroups took 7.9 ms, 30 workgroups 5.8
    with GModelAdapter.Build(with_tables(200, 200, 100, 0.2, 30, 3, 20000), GModelOptions(skip_non_binary=False)) as m:
        init, ms = m.ReadDomains(0), {}
        for _ in range(3):
            for name, run in (("rounds", lambda: m.EnforceGAC(False)), ("block", m.EnforceGAC_Block)):
                m.WriteDomains(0, init)
                ms[name] = min(ms.get(name, 1e9), run().kernel_ms)
    assert ms["rounds"] < 0.43 * ms["block"], ms  # 0.36 spread, 0.49 on two workgroups


@pytest.mark.parametrize("n,d,e,t", [(130, 64, 900, 0.886), (40, 200, 500, 0.95), (20, 1000, 120, 0.985), (70, 3, 1200, 0.05)])
def test_workgroup_seed_with_many_arcs_equals_oracle(gpu, n, d, e, t):
    # the seed's own arcs, 1 to 64 of them per wave, by the wave
    desc = workload.random_binary(n, d, e, t, workload.instance_seed(44, n))
    ok, dom, _ = oracle.Oracle(desc).root_ac()
    assert ok
    deg = np.bincount(desc.con_scope, minlength=n)
    with GModelAdapter.Build(desc) as m:
        for v in (int(np.argmax(deg)), int(np.argmin(deg))):
            vals = domains_to_sets(dom, desc.dom_size)[v]
            for gone in (vals[:1], vals[:len(vals) * 2 // 3]):
                cut = dom.copy()
                for a in gone:
                    cut[v, a // 64] &= ~np.uint64(1 << (a % 64))
                m.WriteDomains(0, cut)
                st = m.EnforceGAC_Block(v)
                ok2, dom2, _ = oracle.Oracle(desc.with_init_dom(cut)).root_ac()
                assert st.inconsistent == (not ok2)
                assert not ok2 or (m.ReadDomains(0) == dom2).all()


def test_workgroup_seed_on_a_tight_network_costs_what_it_does_on_a_loose_one(gpu):
    # one value gone, nothing follows: 16 us either way (142 and 56 with the
    # seed's arcs settled by a lane each)
    ms = {}
    for t in (0.25, 0.886):
        desc = workload.random_binary(2000, 64, 40000, t, 5, preremove=0.05)
        with GModelAdapter.Build(desc) as m:
            assert not m.EnforceGAC(False).inconsistent
            cut = m.ReadDomains(0)
            cut[1000, 0] &= cut[1000, 0] - np.uint64(1)
            for _ in range(3):
                m.WriteDomains(0, cut)
                ms[t] = min(ms.get(t, 1e9), m.EnforceGAC_Block(1000).kernel_ms)
    assert ms[0.886] < 1.8 * ms[0.25], ms


@pytest.mark.parametrize("tables", [8, 16, 17, 32, 33, 64, 65, 200])
def test_tables_in_turn_and_by_changed_variable_equal_oracle(gpu, tables):
    # up to four tables a wave (4 waves in a singleton test, 16 in the others) are
    # taken in turn, more of them by their changed variables
    desc = with_tables(90, 10, 120, 0.35, tables, 3, 200)
    ok, dom, _ = oracle.Oracle(desc, oracle.AC3).root_ac()
    assert ok
    desc = desc.with_init_dom(dom)
    tests = np.array([(v, a) for v, vals in enumerate(domains_to_sets(dom, desc.dom_size)) for a in vals], np.int32)
    want, _ = oracle.Oracle(desc, oracle.AC3).singleton_tests(tests)
    mac = oracle.Oracle(desc, oracle.AC3).mac(node_limit=150, trace_cap=400)
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        got, _ = m.SingletonTests(tests, mode="workgroup")
        assert (got == want).all()
        for v in (int(desc.con_scope[-1]), 3):
            vals = domains_to_sets(dom, desc.dom_size)[v]
            cut = dom.copy()
            cut[v] = np.uint64(1 << vals[0])
            m.WriteDomains(0, cut)
            st = m.EnforceGAC_Block(v)
            ok2, dom2, _ = oracle.Oracle(desc.with_init_dom(cut), oracle.AC3).root_ac()
            assert st.inconsistent == (not ok2)
            assert not ok2 or (m.ReadDomains(0) == dom2).all()
        m.WriteDomains(0, dom)
        st, _, trace = m.Solve(node_limit=150, trace_capacity=400)
        assert trace == mac.trace


@pytest.mark.parametrize("heuristic", ["dom", "dom/wdeg"])
@pytest.mark.parametrize("tables", [64, 65, 200])
@pytest.mark.parametrize("d,arity,tuples,keep", [(12, 3, 700, 0.8), (70, 3, 4000, 0.5)])
def test_searches_over_many_tables_equal_oracle(gpu, d, arity, tuples, keep, tables, heuristic):
    # the search looks at the tables in turn up to four a wave (64), and at the
    # changed ones beyond; small and larger tables
    desc = with_tables(60, d, 50, 0.25, tables, arity, tuples)
    rng = np.random.default_rng(11)
    init = desc.full_domains()
    for v in range(60):
        for a in range(d):
            if rng.random() > keep and a != v % d:
                init[v, a // 64] &= ~np.uint64(1 << (a % 64))
    desc = desc.with_init_dom(init)
    with oracle.var_heuristic(2 if heuristic == "dom/wdeg" else 0):
        want = oracle.Oracle(desc, oracle.AC3).mac(node_limit=60, trace_cap=200)
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        _, _, trace = m.Solve(node_limit=60, trace_capacity=200, heuristic=heuristic)
    assert trace == want.trace


def test_units_over_many_tables_equal_oracle(gpu):
    # units of 16 tables and of more in one launch, at four waves and at sixteen
    descs = [with_tables(60, 12, 50, 0.25, k, 3, 700) for k in (0, 16, 17, 64, 65, 150)]
    want = [oracle.Oracle(desc, oracle.AC3).mac(node_limit=40) for desc in descs]
    try:
        N.tune_set("mac_lds_net", 1)  # (with an image the tables are taken up in turn)
        for threads in (256, 1024):
            N.tune_set("unit_threads", threads)
            res, _ = Batch(descs, GModelOptions(skip_non_binary=False)).run(40)
            for w, r in zip(want, res):
                assert (r.num_positive, r.num_negative) == (w.num_positive, w.num_negative)
    finally:
        N.tune_set("unit_threads", 0)
        N.tune_set("mac_lds_net", 0)


def test_workgroup_passes_over_unchanged_tables(gpu):
    # a value gone from a variable of one table, which loses nothing: one round,
    # whose cost must not grow with the tables of other variables as if they
    # were looked at one after the other (16 waves: 56 turns for 900)
    ms = {}
    for tables in (30, 900):
        desc = with_tables(2000, 12, 100, 0.2, tables, 5, 600)
        count = np.bincount(np.concatenate([s for s in desc.scopes() if len(s) == 5]), minlength=2000)
        v = int(np.flatnonzero(count == 1)[0])
        with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
            assert not m.EnforceGAC(False).inconsistent
            cut = m.ReadDomains(0)
            cut[v, 0] &= cut[v, 0] - np.uint64(1)
            for _ in range(5):
                m.WriteDomains(0, cut)
                st = m.EnforceGAC_Block(v)
                ms[tables] = min(ms.get(tables, 1e9), st.kernel_ms)
            assert st.deletions == 0
    assert ms[900] < 2.0 * ms[30], ms


@pytest.mark.parametrize("mode", ["plain", "persistent", "block"])
@pytest.mark.parametrize("n,d,e,t", [
    # full one-word domains that tight relations leave with many open values:
    # settled by the wave (57 values and 49 open ones are the least)
    (2000, 64, 2000, 0.95), (2000, 64, 1500, 0.97), (60, 64, 60, 0.98), (40, 58, 30, 0.975), (30, 64, 15, 0.97),
])
def test_full_tight_one_word_domains_equal_oracle(gpu, n, d, e, t, mode):
    desc = workload.random_binary(n, d, e, t, 5)
    ok, dom, _ = oracle.Oracle(desc).root_ac()
    with GModelAdapter.Build(desc) as m:
        st = {"plain": lambda: m.EnforceGAC(False), "persistent": lambda: m.EnforceGAC_Persistent(False),
              "block": m.EnforceGAC_Block}[mode]()
        assert st.inconsistent == (not ok)
        assert not ok or (m.ReadDomains(0) == dom).all()


@pytest.mark.parametrize("mode", ["plain", "persistent"])
@pytest.mark.parametrize("n,d,e,t,tables", [
    # the persistent rounds stage up to 128 KB of domains in LDS: 72, 100 and 120
    # KB, and beyond it, where every lane reads memory, with and without tables
    (600, 960, 90, 0.992, 0), (800, 1000, 120, 0.992, 0), (960, 1000, 120, 0.99, 0), (1030, 1000, 150, 0.991, 0),
    (8400, 70, 60, 0.93, 30),
])
def test_staged_and_unstaged_rounds_equal_oracle(gpu, n, d, e, t, tables, mode):
    base = workload.random_binary(n, d, e, t, workload.instance_seed(45, n), preremove=0.1)
    desc = base
    if tables:
        scopes, lists = [list(s) for s in base.scopes()], list(base.tuple_lists())
        rng = np.random.default_rng(n)
        for k in range(tables):
            scopes.append([int(base.con_scope[2 * k]), *map(int, rng.choice(np.arange(n // 2, n), 2, replace=False))])
            lists.append(workload.random_table(500 * n + k, 3, d, 2500))
        desc = from_tuples(base.dom_size, scopes, lists, base.init_dom)
    algo = oracle.AC3 if tables else oracle.AC3BIT
    ok, dom, _ = oracle.Oracle(desc, algo).root_ac()
    assert ok
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        run = (lambda v: m.EnforceGAC(False, v)) if mode == "plain" else (lambda v: m.EnforceGAC_Persistent(False, v))
        st = run(-1)
        assert not st.inconsistent and st.converged
        assert (m.ReadDomains(0) == dom).all()
        removed = 0
        for v in np.argsort(np.bincount(desc.con_scope, minlength=n))[::-1][:3]:  # the best connected ones
            vals = domains_to_sets(dom, desc.dom_size)[v]
            cut = dom.copy()
            for a in vals[::2]:
                cut[v, a // 64] &= ~np.uint64(1 << (a % 64))
            m.WriteDomains(0, cut)
            st = run(int(v))
            ok2, dom2, _ = oracle.Oracle(desc.with_init_dom(cut), algo).root_ac()
            assert st.inconsistent == (not ok2)
            if ok2:
                assert (m.ReadDomains(0) == dom2).all()
                removed += int(np.bitwise_count(cut).sum()) - int(np.bitwise_count(dom2).sum())
        assert removed > 0, "the seeded half removed nothing"

"""Seeded fixpoints on levels that are not at their closure (needs an MI355X).

EnforceGAC(assigned_var) propagates from one variable.  On a level whose other
variables also lost values (by RemoveValue or WriteDomains) what it reaches
depends on what it looks at again, and that is part of each mode's answer:

* host-driven, persistent, allocation-free and asynchronous fixpoints keep a
  frontier of constraints, as GModel::EnforceGAC does (src/GModel.cu:1110-1220):
  every position of a constraint is revised once one of its variables changed;
* the workgroup fixpoint and the singleton tests keep a frontier of variables, as
  AC3 does (src/AC3.cpp:99-141): a position is revised once another of the
  constraint's variables changed; a seeded fixpoint revises every position of
  the seed's constraints too.

Both closures are unique, so a plain restatement of each is the oracle.
"""
import ctypes as C

import numpy as np
import pytest

from cpim_amd import GModelAdapter, GModelOptions, workload
from cpim_amd import _native as N
from cpim_amd.model import domains_to_sets, from_tuples

pytestmark = pytest.mark.gpu


def seeded_closure(desc, sets, seed, frontier):
    """The domains after propagation from `seed` (None: a wipe-out).  frontier:
    "constraint", "variable", or "assigned" (of variables, and the seed is a
    decision, which is not revised)."""
    scopes, lists = [list(map(int, s)) for s in desc.scopes()], desc.tuple_lists()
    of = [[] for _ in range(desc.num_vars)]
    for c, s in enumerate(scopes):
        for v in s:
            of[v].append(c)
    dom = [set(s) for s in sets]
    moved = {seed}

    def revised(s, v):
        if frontier == "constraint" or any(u in moved for u in s if u != v):
            return v != seed or frontier != "assigned"
        return frontier == "variable" and seed in s

    todo = list(of[seed])
    while todo:
        c = todo.pop()
        s, t = scopes[c], np.asarray(lists[c])
        valid = t[np.all([np.isin(t[:, p], list(dom[v])) for p, v in enumerate(s)], axis=0)]
        for p, v in enumerate(s):
            keep = dom[v] & set(valid[:, p].tolist())
            if keep != dom[v] and revised(s, v):
                if not keep:
                    return None
                dom[v] = keep
                moved.add(v)
                todo += [k for k in of[v] if k not in todo]
    return dom


def network(n, d, e, t, tables, seed, tuples=0):
    base = workload.random_binary(n, d, e, t, workload.instance_seed(41, seed))
    scopes, lists = [list(s) for s in base.scopes()], list(base.tuple_lists())
    rng = np.random.default_rng(seed)
    for k in range(tables):
        at = int(rng.integers(0, len(scopes) + 1))
        scopes.insert(at, rng.choice(n, 3, replace=False).tolist())
        lists.insert(at, workload.random_table(4100 * seed + k, 3, d, tuples))
    # some values of every variable gone
    sets = [set(np.flatnonzero(rng.random(d) < 0.8).tolist()) or {0} for _ in range(n)]
    return from_tuples(base.dom_size, scopes, lists), sets


def words(sets, W):
    out = np.zeros((len(sets), W), np.uint64)
    for v, s in enumerate(sets):
        for a in s:
            out[v, a // 64] |= np.uint64(1 << (a % 64))
    return out


def noalloc(m, v):
    st = N.CGacStats()
    N.check(N.gpu_lib().cpim_gmodel_enforce_gac_noalloc(m.handle, v, C.byref(st)))
    return st


MODES = {
    "plain": ("constraint", lambda m, v: m.EnforceGAC(False, v)),
    "persistent": ("constraint", lambda m, v: m.EnforceGAC_Persistent(False, v)),
    "noalloc": ("constraint", noalloc),
    "async": ("constraint", lambda m, v: m.EnforceGAC_Async(v)),
    "block": ("variable", lambda m, v: m.EnforceGAC_Block(v)),
    # of variables up to 4,096 constraints, whichever kernel runs
    "auto": (None, lambda m, v: m.EnforceGAC_Auto(v)),
}

# n, d, e, t, tables, tuples: one and two words, small tables and larger ones,
# and 300, 1,000 and 4,200 constraints
SHAPES = [
    (60, 8, 90, 0.55, 0, 0), (60, 8, 90, 0.45, 20, 60), (40, 70, 60, 0.925, 0, 0), (40, 20, 40, 0.72, 14, 400),
    (200, 6, 1000, 0.30, 0, 0), (200, 6, 950, 0.26, 60, 70), (600, 6, 4200, 0.27, 0, 0),
]


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_seeded_fixpoint_on_an_open_level(gpu, shape, mode):
    n, d, e, t, tables, tuples = shape
    frontier, run = MODES[mode]
    if frontier is None:
        frontier = "constraint" if e + tables > 4096 else "variable"
    other = 0  # seeds on which the other frontier's closure is another one
    for seed in range(4):
        desc, sets = network(n, d, e, t, tables, seed, tuples)
        v = int(np.random.default_rng(seed).integers(0, n))
        sets[v] = set(sorted(sets[v])[::2]) if d > 64 else {min(sets[v])}
        want = seeded_closure(desc, sets, v, frontier)
        other += want != seeded_closure(desc, sets, v, "variable" if frontier == "constraint" else "constraint")
        with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
            m.WriteDomains(0, words(sets, m.dom_words))
            st = run(m, v)
            assert bool(st.inconsistent) == (want is None), seed
            if want is not None:
                got = domains_to_sets(m.ReadDomains(0), desc.dom_size)
                assert [set(g) for g in got] == want, seed
    assert other, "the two frontiers agree on every seed: the shape tests nothing"


@pytest.mark.parametrize("shape", [s for s in SHAPES if s[2] < 1000], ids=str)
def test_workgroup_singleton_tests_on_an_open_level(gpu, shape):
    n, d, e, t, tables, tuples = shape
    desc, sets = network(n, d, e, t, tables, 1, tuples)
    tests = [(v, a) for v, s in enumerate(sets) for a in sorted(s)][::max(1, n * d // 150)]
    want = [seeded_closure(desc, sets[:v] + [{a}] + sets[v + 1:], v, "assigned") is None for v, a in tests]
    with GModelAdapter.Build(desc, GModelOptions(skip_non_binary=False)) as m:
        m.WriteDomains(0, words(sets, m.dom_words))
        got, _ = m.SingletonTests(np.array(tests, np.int32), mode="workgroup")
    assert got.astype(bool).tolist() == want


@pytest.mark.parametrize("shape", [(60, 8, 90, 0.6), (60, 8, 100, 0.6), (80, 6, 140, 0.5), (50, 30, 90, 0.85)], ids=str)
def test_auto_singleton_tests_on_an_open_level(gpu, shape):
    """Binary networks: on an open level a bit-sliced test sees what the other
    tests of its group revise as well, so which tests fail depends on the
    kernel, and the automatic choice stays with the bit-sliced one there."""
    n, d, e, t = shape
    desc, sets = network(n, d, e, t, 0, 1)
    tests = np.array([(v, a) for v, s in enumerate(sets) for a in sorted(s)], np.int32)
    with GModelAdapter.Build(desc) as m:
        m.WriteDomains(0, words(sets, m.dom_words))
        got = {mode: m.SingletonTests(tests, mode=mode)[0] for mode in ("auto", "sliced", "workgroup")}
        assert (got["sliced"] != got["workgroup"]).any(), "the two kernels agree: the shape tests nothing"
        assert (got["auto"] == got["sliced"]).all()

"""Automatic choices between kernels, where the wrong one costs several times
the right one (needs an MI355X)."""
import numpy as np
import pytest

from cpim_amd import GModelAdapter, workload
from cpim_amd.model import ModelDesc, domains_to_sets, words_for

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

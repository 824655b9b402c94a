"""Pools that take over the buffers of earlier pools of their graph: the same
sets and seeds as on fresh buffers, from several threads, and the memory back
when the graph goes."""
import ctypes as C
import threading

import numpy as np
import pytest

import ripples_amd as R

pytestmark = pytest.mark.gpu


def rmat_graph(scale, scheme, wscale, seed, model):
    s, d = R.rmat_edges(scale, seed=seed)
    index, edges, w = R.csr_from_edges(1 << scale, s, d, scheme, wscale, seed)
    return index, edges, w, R.Graph(index, edges, w, model=model)


def device_free():
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


GRAPHS = {
    "cascade": (13, R.W_CASCADE, 1.0, 3, R.IC),    # plain pools
    "uniform": (13, R.W_UNIFORM, 0.1, 4, R.IC),    # columns
    "lt": (13, R.W_LT_NORM, 0.9, 5, R.LT),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_pools_after_pools_match_oracle(name, orc):
    index, edges, w, g = rmat_graph(*GRAPHS[name])
    model, n = GRAPHS[name][-1], len(index) - 1
    # growing, shrinking, equal, and one that grows in steps
    for i, counts in enumerate([[3000], [500], [3000], [100, 700, 1, 1500], [64], [2000]]):
        p = g.pool(40 + i)
        for c in counts:
            p.generate_rrr_sets(c)
        off, ver = p.export()
        eo, ev = orc.sample(model, index, edges, w, 40 + i, 0, sum(counts))
        assert np.array_equal(off, eo) and np.array_equal(ver, ev)
        seeds, cov = p.find_most_influential_set(5)
        es, ec = orc.select(n, eo, ev, 5)
        assert seeds.tolist() == es.tolist() and cov == ec
        assert np.array_equal(p.count_occurrences(), orc.count(n, eo, ev))
        p.close()
    g.close()


def test_threads_share_a_graphs_blocks():
    index, edges, w, g = rmat_graph(13, R.W_UNIFORM, 0.1, 6, R.IC)

    def one(seed):
        p = g.pool(seed)
        p.generate_rrr_sets(400 + 300 * (seed % 4))
        off, ver = p.export()
        seeds, cov = p.find_most_influential_set(4)
        p.close()
        return off.tolist(), ver.tolist(), seeds.tolist(), cov

    want = {s: one(s) for s in range(8)}
    got = {}

    def work(seeds):
        for s in seeds:
            got[s] = one(s)

    for _ in range(3):
        ts = [threading.Thread(target=work, args=(range(t, 8, 4),)) for t in range(4)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert got == want
        got.clear()
    g.close()


def test_memory_comes_back():
    free = []
    for _ in range(3):
        index, edges, w, g = rmat_graph(14, R.W_UNIFORM, 0.1, 7, R.IC)
        for count in (1000, 8000, 3000):
            p = g.pool(1)
            p.generate_rrr_sets(count)
            p.find_most_influential_set(3)
            p.close()
        g.close()
        free.append(device_free())
    assert free[2] >= free[0] - (32 << 20)   # what the runtime itself keeps

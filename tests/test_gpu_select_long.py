"""Selection of plain pools of long sets against the oracle: rounds that turn to
the whole GPU by the members of a list and not by its sets, and pools of more than
2^23 members that end in the full index sorted by vertex."""
import ctypes as C

import numpy as np
import pytest

import ripples_amd as R

pytestmark = pytest.mark.gpu


def drawn(n, count, low, high, power, seed):
    """Sets of low..high draws, vertices skewed by the power."""
    rng = np.random.default_rng(seed)
    return n, [np.unique((n * rng.random(rng.integers(low, high + 1)) ** power).astype(np.int64))
               for _ in range(count)]


def cliques(n, count, size, copies):
    """Vertices that share all their sets: a pass over the pool yields one round."""
    return n, [np.arange(c * size, (c + 1) * size) for c in range(count) for _ in range(copies - c)]


# below and above 4 x 32,768 members and 4,096 sets; lists either side of the
# line, which lies at 32,768 members
POOLS = {
    "few short": lambda: drawn(900, 600, 150, 210, 2, 1),
    "few": lambda: drawn(900, 1000, 250, 350, 2, 2),
    "even": lambda: drawn(3000, 3000, 200, 400, 1, 3),
    "many": lambda: drawn(1500, 6000, 100, 300, 2, 4),
    "most": lambda: drawn(400, 5000, 300, 900, 1, 5),
    "cliques": lambda: cliques(60000, 20, 1100, 60),
    "one": lambda: (70000, [np.arange(0, 70000, 2)]),
}


def filled(n, sets):
    off = np.zeros(len(sets) + 1, np.uint64)
    off[1:] = np.cumsum([len(s) for s in sets])
    ver = np.concatenate(sets).astype(np.uint32)
    g = R.Graph(np.zeros(n + 1, np.uint64), np.zeros(0, np.uint32), np.zeros(0, np.float32))
    p = g.pool(0)
    p.append(off, ver)
    return off, ver, g, p


def device_free():
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("name", sorted(POOLS))
def test_long_sets_match_oracle(name, orc):
    n, sets = POOLS[name]()
    off, ver, g, p = filled(n, sets)
    assert np.array_equal(p.count_occurrences(), orc.count(n, off, ver))
    for k in (1, 12, 150):
        seeds, cov = p.find_most_influential_set(k)
        es, ec = orc.select(n, off, ver, k)
        assert seeds.tolist() == es.tolist() and cov == ec
    p.close()
    g.close()


# the search among candidates gives up after two seeds, and before the first
# (more vertices of the largest count than it takes, that count past 127)
@pytest.mark.parametrize("pool", [(1100000, 20, 4000, 120), (400000, 14, 1100, 560)])
def test_sorted_index_matches_oracle(pool, orc):
    n, sets = cliques(*pool)
    off, ver, g, p = filled(n, sets)
    total = int(off[-1])
    assert total >= 1 << 23
    before = device_free()
    for k in (1, 2, 3, 40):
        seeds, cov = p.find_most_influential_set(k)
        es, ec = orc.select(n, off, ver, k)
        assert seeds.tolist() == es.tolist() and cov == ec
    # lists (4 bytes a member), buckets and candidates (2 each), and the pairs
    # of the sort: 12 more
    assert before - device_free() > 16 * total
    p.close()
    g.close()


def test_more_seeds_than_a_graph_holds(orc):
    """A pool with column sets, whose rounds run over all vertices."""
    src, dst = R.rmat_edges(14, seed=9)
    index, edges, w = R.csr_from_edges(1 << 14, src, dst, R.W_UNIFORM, 0.1, 9)
    g = R.Graph(index, edges, w)
    p = g.pool(5)
    p.generate_rrr_sets(20000)
    assert p.columns()[0] > 0
    off, ver = p.export()
    for k in (4096, 4097, 6000):
        seeds, cov = p.find_most_influential_set(k)
        es, ec = orc.select(1 << 14, off, ver, k)
        assert seeds.tolist() == es.tolist() and cov == ec
    p.close()
    g.close()

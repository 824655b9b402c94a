"""Selection of plain pools among the vertices of largest count, on pools
where its rules can go wrong, against the oracle: seeds, coverage, counts."""
import numpy as np
import pytest

import ripples_amd as R

pytestmark = pytest.mark.gpu


def csr(sets):
    off = np.zeros(len(sets) + 1, np.uint64)
    off[1:] = np.cumsum([len(s) for s in sets])
    return off, (np.concatenate(sets) if sets else np.zeros(0)).astype(np.uint32)


def singles(n):
    """Every vertex in one set: one count, far more vertices than candidates."""
    return n, [np.array([v]) for v in range(n)]


def flat(n, count, seed):
    """Counts of a few, most of them equal."""
    rng = np.random.default_rng(seed)
    return n, [np.unique(rng.integers(0, n, rng.integers(0, 3))) for _ in range(count)]


def clusters(k, size, copies):
    """Vertices that share all their sets: each seed empties a cluster."""
    return k * size, [np.arange(c * size, (c + 1) * size) for c in range(k) for _ in range(copies - c)]


def regular(n, times, width, seed):
    """Every vertex in exactly `times` sets: no bin of large counts fits."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(times):
        p = rng.permutation(n)
        out += [np.sort(x) for x in np.split(p, range(width, n, width))]
    return n, out


def skewed(n, count, mean, seed):
    """Hubs in tens of thousands of sets beside vertices in one."""
    rng = np.random.default_rng(seed)
    size = rng.poisson(mean, count)
    v = (n * rng.random(int(size.sum())) ** 6).astype(np.int64)
    return n, [np.unique(x) for x in np.split(v, np.cumsum(size)[:-1])]


POOLS = {
    "singles": lambda: singles(10001),
    "flat": lambda: flat(20000, 30000, 1),
    "tiny": lambda: flat(3, 9, 2),
    "clusters": lambda: clusters(14, 5000, 20),
    "regular": lambda: regular(6000, 200, 6, 3),
    "skewed": lambda: skewed(70001, 90000, 8, 4),
}


@pytest.mark.parametrize("name", sorted(POOLS))
def test_selection_matches_oracle(name, orc):
    n, sets = POOLS[name]()
    off, ver = csr(sets)
    g = R.Graph(np.zeros(n + 1, np.uint64), np.zeros(0, np.uint32), np.zeros(0, np.float32))
    p = g.pool(0)
    p.append(off, ver)
    for num in (len(sets), len(sets) // 3, 1):
        part = ver[:int(off[num])]
        assert np.array_equal(p.count_occurrences(num), orc.count(n, off[:num + 1], part))
        for k in (1, 60, 200):
            seeds, cov = p.find_most_influential_set(k, num)
            es, ec = orc.select(n, off[:num + 1], part, k)
            assert seeds.tolist() == es.tolist() and cov == ec
    p.close()
    g.close()

"""Selection of plain pools of long sets, whose rounds turn to the whole GPU by
the members of a list and not by its sets, against the oracle."""
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


@pytest.mark.parametrize("name", sorted(POOLS))
def test_long_sets_match_oracle(name, orc):
    n, sets = POOLS[name]()
    off = np.zeros(len(sets) + 1, np.uint64)
    off[1:] = np.cumsum([len(s) for s in sets])
    ver = np.concatenate(sets).astype(np.uint32)
    g = R.Graph(np.zeros(n + 1, np.uint64), np.zeros(0, np.uint32), np.zeros(0, np.float32))
    p = g.pool(0)
    p.append(off, ver)
    assert np.array_equal(p.count_occurrences(), orc.count(n, off, ver))
    for k in (1, 12, 150):
        seeds, cov = p.find_most_influential_set(k)
        es, ec = orc.select(n, off, ver, k)
        assert seeds.tolist() == es.tolist() and cov == ec
    p.close()
    g.close()

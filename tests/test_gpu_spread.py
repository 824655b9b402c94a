"""The spread simulator's kernels against the oracle, replica by replica: few
and many replicas (the workgroup sizes), bitmaps in LDS and in device memory,
long rows, sums that meet their threshold exactly, irregular weights."""
import numpy as np
import pytest

import ripples_amd as R

pytestmark = pytest.mark.gpu


def rmat(n, scale, ef, scheme, wscale, seed):
    s, d = R.rmat_edges(scale, ef, seed=seed)
    s, d = s.astype(np.int64) % n, d.astype(np.int64) % n
    key = np.unique((s * n + d)[s != d])
    return R.csr_from_edges(n, (key // n).astype(np.uint32), (key % n).astype(np.uint32), scheme,
                            wscale, seed)


def check(model, csr, seeds, count, orc):
    index, edges, w = csr
    g = R.Graph(index, edges, w, model=model)
    act, lev = g.spread(seeds, count, seed=9, first=7)
    ea, el = orc.spread(model, index, edges, w, seeds, 9, 7, count)
    assert np.array_equal(act, ea) and np.array_equal(lev, el)
    g.close()


@pytest.mark.parametrize("count", [1, 5, 300, 1100])
def test_replicas_match_oracle(count, orc):
    seeds = np.arange(12, dtype=np.uint32)
    check(R.IC, rmat(5003, 13, 16, R.W_UNIFORM, 0.2, 1), seeds, count, orc)
    check(R.LT, rmat(5003, 13, 16, R.W_LT_NORM, 0.95, 2), seeds, count, orc)


@pytest.mark.parametrize("n", [(1 << 19) + 1, (1 << 20) + 1])   # past LT's bitmaps, past IC's
def test_bitmaps_in_memory_match_oracle(n, orc):
    seeds = np.arange(64, dtype=np.uint32)
    check(R.IC, rmat(n, 20, 2, R.W_UNIFORM, 0.9, 3), seeds, 6, orc)
    check(R.LT, rmat(n, 20, 2, R.W_LT_NORM, 0.95, 4), seeds, 6, orc)


def test_lt_sums_at_the_threshold(orc):
    """In-weights of 2^-24 multiples that add up to values thresholds take,
    where only the ordered float sum can decide; and rows with negative,
    infinite or NaN weights."""
    rng = np.random.default_rng(5)
    index, edges, w = rmat(2000, 11, 16, R.W_LT_NORM, 1.0, 5)
    coarse = (np.ceil(w * 16) / 16).astype(np.float32)
    check(R.LT, (index, edges, coarse), np.arange(9, dtype=np.uint32), 200, orc)
    third = np.where(w > 0.02, np.float32(1 / 3), np.float32(1e-7)).astype(np.float32)
    check(R.LT, (index, edges, third), np.arange(9, dtype=np.uint32), 200, orc)
    odd = w.copy()
    hit = rng.random(len(odd)) < 0.02
    odd[hit] = rng.choice(np.array([-0.5, np.inf, np.nan, -np.inf], np.float32), hit.sum())
    check(R.LT, (index, edges, odd), np.arange(9, dtype=np.uint32), 200, orc)


@pytest.mark.parametrize("wscale", [0.2, 0.5, 0.8])
def test_lt_replicas_one_after_the_other(wscale, orc):
    """Several replicas to a workgroup, whose sums start at zero whether the one
    before met few edges or many."""
    seeds = np.arange(0, 40, 2, dtype=np.uint32)
    check(R.LT, rmat(3001, 12, 6, R.W_LT_NORM, wscale, 5), seeds, 4000, orc)
    check(R.LT, rmat(40009, 16, 8, R.W_LT_NORM, wscale, 6), seeds[:4], 2500, orc)


def test_lt_calls_one_after_the_other(orc):
    """Calls on one graph that leave sums behind and calls that do not."""
    index, edges, w = rmat(9001, 14, 8, R.W_LT_NORM, 0.9, 7)
    g = R.Graph(index, edges, w, model=R.LT)
    many, few = np.arange(400, dtype=np.uint32), np.array([8999], np.uint32)
    for seeds, count in ((many, 40), (few, 60), (many, 3), (few, 2), (many, 1500), (few, 1500), (many, 30)):
        act, lev = g.spread(seeds, count, seed=11)
        ea, el = orc.spread(R.LT, index, edges, w, seeds, 11, 0, count)
        assert np.array_equal(act, ea) and np.array_equal(lev, el)
    g.close()

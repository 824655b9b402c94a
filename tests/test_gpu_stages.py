"""AUTO's automatic setting through the C ABI: calls either side of the size
that takes the lanes, on graphs whose rows have one gap block (weighted
cascade), several (U[0,0.1], hubs of hundreds) and none."""
import numpy as np
import pytest

import ripples_amd as R
from graphs import transposed_csr

pytestmark = pytest.mark.gpu


def rmat_csr(scale, scheme, wscale, seed):
    s, d = R.rmat_edges(scale, seed=seed)
    return R.csr_from_edges(1 << scale, s, d, scheme, wscale, seed)


GRAPHS = {
    "cascade": lambda: rmat_csr(12, R.W_CASCADE, 1.0, 4),
    "uniform": lambda: rmat_csr(12, R.W_UNIFORM, 0.1, 5),
    "certain": lambda: rmat_csr(8, R.W_CONST, 1.0, 6),       # T = 2^24: every candidate, gap 0
    "dead": lambda: rmat_csr(8, R.W_CONST, 1e-9, 7),            # thresholds 0: no live edge
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
@pytest.mark.parametrize("count", [1, 63, 64, 65, 4096, 4097, 16385])
def test_automatic_setting_matches_oracle(name, count, orc):
    index, edges, w = GRAPHS[name]()
    g = R.Graph(index, edges, w, model=R.IC)
    p = g.pool(21)
    p.generate_rrr_sets(count)
    part = min(count, 3000)
    for first in {0, count - part}:
        off, ver = p.export(first, part)
        eo, ev = orc.sample(R.IC, index, edges, w, 21, first, part)
        assert np.array_equal(off, eo) and np.array_equal(ver, ev)
    p.close()
    g.close()


def folded_csr(n, scale, edge_factor, scheme, wscale, seed):
    """R-MAT edges folded onto n vertices (any number of them)."""
    s, d = R.rmat_edges(scale, edge_factor, seed=seed)
    s, d = s.astype(np.int64) % n, d.astype(np.int64) % n
    key = np.unique((s * n + d)[s != d])
    return R.csr_from_edges(n, (key // n).astype(np.uint32), (key % n).astype(np.uint32), scheme,
                            wscale, seed)


@pytest.mark.parametrize("n,scale,ef,wscale,count", [
    (65, 8, 8, 0.4, 700),             # bitmaps of three words, one hot vertex per lane
    (1000, 10, 8, 0.3, 900),
    (4097, 12, 16, 0.1, 257),         # more samples than CUs: workgroups of 512
    (32768, 15, 16, 0.1, 200),
    (70001, 16, 16, 0.1, 1500),       # many samples: workgroups of 256, columns
    (262147, 18, 8, 0.2, 150),        # bitmaps past 32 KiB
    (1 << 20, 20, 4, 0.5, 70),        # the largest bitmap
    ((1 << 20) + 1, 20, 4, 0.5, 70),  # one vertex more: the grid sampler
])
def test_team_sampler_matches_oracle(n, scale, ef, wscale, count, orc):
    """Samples past 64 vertices straight to a workgroup each; in two calls, so
    the second appends and its groups are ragged."""
    index, edges, w = folded_csr(n, scale, ef, R.W_UNIFORM, wscale, n)
    g = R.Graph(index, edges, w, model=R.IC)
    p = g.pool(5)
    for c in (count // 3, count - count // 3):
        p.generate_rrr_sets(c, tune={"queue_cap": 64})
    off, ver = p.export()
    eo, ev = orc.sample(R.IC, index, edges, w, 5, 0, count)
    assert np.array_equal(off, eo) and np.array_equal(ver, ev)
    assert p.size() == (count, len(ev))
    assert np.array_equal(p.count_occurrences(), orc.count(n, eo, ev))
    seeds, cov = p.find_most_influential_set(8)
    es, ec = orc.select(n, eo, ev, 8)
    assert seeds.tolist() == es.tolist() and cov == ec
    p.close()
    g.close()


def hubs_csr(deg):
    """100 hubs that every other vertex has as in-neighbours, each with `deg`
    in-edges, one of threshold 2^23 (blocks of 16 edges) and the rest next to
    dead."""
    n = 3000 + deg
    hubs, rest = np.arange(100), np.arange(100, n)
    s = [np.tile(hubs, len(rest))]
    d = [np.repeat(rest, 100)]
    w = [np.ones(100 * len(rest), np.float32)]
    for h in hubs:
        s.append(100 + (np.arange(deg) * 7 + 31 * h) % (deg + 1000))
        d.append(np.full(deg, h))
        w.append(np.full(deg, 1e-5, np.float32))
        w[-1][(17 * h) % deg] = 0.5
    return transposed_csr(n, np.concatenate(s), np.concatenate(d), np.concatenate(w))


@pytest.mark.parametrize("deg,count,cap", [
    (511, 64 * 3 + 5, 0),         # thin frontiers, rows next to the size that is cut up
    (513, 64 * 3 + 5, 0),
    (513, 64 * 200 + 1, 0),       # wide ones: hub rows of 2112 units in segments
    (512, 64 * 200 + 1, 37),      # no room for most of the segments, nor the frontier
    (16003, 64 * 3 + 5, 100),     # 64 segments a row
])
def test_grid_sampler_hub_rows_match_oracle(deg, count, cap, orc):
    index, edges, w = hubs_csr(deg)
    g = R.Graph(index, edges, w, model=R.IC)
    p = g.pool(9)
    p.generate_rrr_sets(count, tune={"queue_cap": 64, "colors": 64, "frontier_cap": cap})
    for first in {0, max(0, count - 600)}:
        part = min(count, 600)
        off, ver = p.export(first, part)
        eo, ev = orc.sample(R.IC, index, edges, w, 9, first, part)
        assert np.array_equal(off, eo) and np.array_equal(ver, ev)
    p.close()
    g.close()


def cycles_csr(lengths, reps, isolated):
    """Cycles whose edges are all live in both directions (a set is its root's
    whole cycle) and isolated vertices."""
    s, d, at = [], [], 0
    for length in np.tile(lengths, reps):
        v = at + np.arange(length)
        u = at + (np.arange(length) + 1) % length
        s += [v, u]
        d += [u, v]
        at += length
    s, d = np.concatenate(s), np.concatenate(d)
    return transposed_csr(at + isolated, s, d, np.ones(len(s), np.float32))


SHORT = [3, 15, 16, 17, 18, 31, 63, 64, 65, 66, 95, 96, 97, 127, 128, 129, 255, 256, 257]
LONG = SHORT + [191, 192, 193, 383, 384, 385, 511, 512, 513, 767, 768, 769, 1023, 1024, 1025]
WIDE = LONG + [1535, 1536, 2047, 2048, 2049, 4095, 4096, 4097]


@pytest.mark.parametrize("lengths,reps,isolated,count", [
    (LONG, 3, 100, 1),
    (LONG, 3, 100, 4096),              # a sample per wave
    (LONG, 3, 100, 4097),              # lanes first from here on
    (LONG, 3, 100, 19000),             # two per wave
    (SHORT, 40, 100, 45000),           # lanes first, four per wave behind them
    (WIDE, 6, 1 << 20, 1500),          # past 2^20 vertices: sets of up to 4096
    (WIDE, 6, 1 << 20, 17000),
])
def test_wave_stage_set_lengths_match_oracle(lengths, reps, isolated, count, orc):
    index, edges, w = cycles_csr(lengths, reps, isolated)
    g = R.Graph(index, edges, w, model=R.IC)
    p = g.pool(3)
    for first in (0, count):           # the second call finds the scratch of the first
        p.generate_rrr_sets(count)
        off, ver = p.export(first, count)
        eo, ev = orc.sample(R.IC, index, edges, w, 3, first, count)
        assert np.array_equal(off, eo) and np.array_equal(ver, ev)
    p.close()
    g.close()

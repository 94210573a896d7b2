"""Induced bit matrices and outside rows at the edges of the list walk: lists
of few and of many arcs, shorter and longer than a wave takes at a time, vs the
CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bipartite(a, b, extra, seed):
    """K(a, b) and `extra` random edges inside the larger side: out-lists of
    about min(a, b) arcs."""
    u = np.repeat(np.arange(a), b)
    v = a + np.tile(np.arange(b), a)
    rng = np.random.default_rng(seed)
    eu = a + rng.integers(0, b, extra)
    ev = a + rng.integers(0, b, extra)
    keep = eu != ev
    return np.concatenate([u, eu[keep]]), np.concatenate([v, ev[keep]]), a + b


@pytest.mark.parametrize("a,b,extra", [(3, 700, 40), (15, 64, 30), (63, 66, 50), (64, 64, 0), (65, 130, 60),
                                       (127, 140, 40), (255, 256, 30), (256, 257, 30), (257, 300, 60)])
def test_lists_of_all_lengths(mce, oracle, a, b, extra):
    u, v, n = bipartite(a, b, extra, 11)
    g = mce.from_edges(u, v, n=n)
    with mce.DeviceGraph(g) as dg:
        dg.order()
        for level in (1, 2):
            ref = oracle.mce(g, level=level, ipx=True)
            for opts in ({}, {"lds_arena_bytes": 1024}, {"lane_universe": -1, "small_universe": -1}):
                print(f"case {a} {b} level={level} {opts}", flush=True)
                res = dg.count(level=level, induced=2, worklist=1, **opts)
                for k in ("count", "hist", "hash", "tree_nodes"):
                    assert res[k] == ref[k], (k, opts)


@pytest.mark.parametrize("a,b,extra", [(20, 90, 300), (257, 300, 400), (1030, 1040, 500)])
def test_features_count_inner_edges(mce, a, b, extra):
    # up to and past the members that a wave keeps in LDS (1,024)
    u, v, n = bipartite(a, b, extra, 5)
    g = mce.from_edges(u, v, n=n)
    with mce.DeviceGraph(g) as dg:
        dg.order()
        F = dg.features()
        _, split, oc = dg.download()
    rp = g.row_ptr.astype(np.int64)
    split = split.astype(np.int64)
    deg = rp[1:] - split
    for x in list(np.argsort(-deg)[:6]) + list(range(0, n, max(n // 20, 1))):
        P = oc[split[x]:rp[x + 1]]
        inner = sum(int(np.isin(oc[split[w]:rp[w + 1]], P).sum()) for w in P)
        assert abs(F[x, 7] - np.log1p(inner)) <= 1e-5 * max(1.0, np.log1p(inner))

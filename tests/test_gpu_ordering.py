"""Degeneracy ordering on the GPU at the sizes where its route changes: one
workgroup with row offsets in LDS (up to 16,384 vertices), without them (up to
32,768), and the grid with a one-workgroup tail; arcs above what one workgroup
takes; frontiers longer than their LDS part; rows long enough for the whole
workgroup, and more of them than its list holds; levels with no round."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def matching_and_clique(mce, n, k):
    """A perfect matching on n - k vertices and a clique on the last k."""
    a = np.arange(0, n - k - 1, 2)
    iu = np.triu_indices(k, 1)
    return mce.from_edges(np.concatenate([a, iu[0] + n - k]), np.concatenate([a + 1, iu[1] + n - k]), n=n)


def bipartite(mce, a, b):
    x, y = np.meshgrid(np.arange(a), np.arange(b), indexing="ij")
    return mce.from_edges(x.ravel(), y.ravel() + a, n=a + b)


def hubs(mce, n, k):
    """k hubs joined to every vertex, the rest a path."""
    h, v = np.meshgrid(np.arange(k), np.arange(k, n), indexing="ij")
    p = np.arange(k, n - 1)
    return mce.from_edges(np.concatenate([h.ravel(), p]), np.concatenate([v.ravel(), p + 1]), n=n)


CASES = {
    "er16384": lambda m: m.gen_er(16384, 60000, 1),
    "er16385": lambda m: m.gen_er(16385, 60000, 2),
    "er32768": lambda m: m.gen_er(32768, 150001, 3),
    "er32769": lambda m: m.gen_er(32769, 150001, 4),
    "matching": lambda m: matching_and_clique(m, 20000, 61),
    "matching-large": lambda m: matching_and_clique(m, 90000, 300),
    "bipartite-many-long-rows": lambda m: bipartite(m, 600, 601),
    "bipartite-arcs": lambda m: bipartite(m, 1100, 1101),
    "hubs": lambda m: hubs(m, 30000, 5),
    "hubs-large": lambda m: hubs(m, 70001, 3),
    "dense-arcs": lambda m: m.gen_rmat(12, 250, seed=5),
    "rmat16": lambda m: m.gen_rmat(16, 16, seed=6),
    "chung-lu": lambda m: m.gen_chung_lu(100003, 2.1, 24.0, 48, 20, 60, seed=7),
    "sbm-batch": lambda m: m.gen_sbm_batch(200, 64, 700, seed=8)[1],
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_order_matches_oracle(mce, oracle, name):
    g = CASES[name](mce)
    prio_o, split_o, oc_o, degen = oracle.order_orient(g)
    with mce.DeviceGraph(g) as dg:
        for k in range(2):  # a second ordering of the same graph starts afresh
            info = dg.order()
            prio, split, oc = dg.download()
            assert info["degeneracy"] == degen
            np.testing.assert_array_equal(prio, prio_o)
            np.testing.assert_array_equal(split, split_o)
            np.testing.assert_array_equal(oc, oc_o)
    deg = g.degrees()
    assert info["max_degree"] == deg.max()
    assert info["max_out_degree"] == (g.row_ptr[1:].astype(np.int64) - split_o.astype(np.int64)).max()

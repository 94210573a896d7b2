"""Lane solver (one subtree per lane, 64 queued per wave) and donation at the
engine's own thresholds vs the CPU oracle: bit-exact totals and per-subproblem
labels where the queue's limits bind."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def union(mce, parts):
    """Disjoint union of graphs given as (n, u, v)."""
    base, us, vs = 0, [], []
    for n, u, v in parts:
        us.append(u + base)
        vs.append(v + base)
        base += n
    return mce.from_edges(np.concatenate(us), np.concatenate(vs), n=base)


def dense(n, p, seed):
    u, v = np.triu_indices(n, 1)
    keep = np.random.default_rng(seed).random(u.size) < p
    return n, u[keep], v[keep]


def multipartite(parts, size):
    """Complete multipartite graph: every pivot score is a tie."""
    n = parts * size
    u, v = np.triu_indices(n, 1)
    keep = u // size != v // size
    return n, u[keep], v[keep]


GRAPHS = {
    # universes of 10..66 members: |P| and |X| on both sides of 15 and 16,
    # 16 and 17 (second column word), 48 and 49, 64 and 65
    "sizes": lambda mce: union(mce, [dense(n, p, 97 * n + int(10 * p)) for n in range(10, 67, 2)
                                     for p in (0.3, 0.6, 0.8)]),
    "ties": lambda mce: union(mce, [multipartite(k, s) for k, s in
                                    ((15, 1), (16, 1), (17, 1), (49, 1), (8, 2), (12, 2), (6, 3), (7, 3), (4, 5), (3, 16))]),
    # few large trees: full queues inside a subtree, cliques past the buffer
    "large": lambda mce: union(mce, [dense(150, 0.6, 3), dense(130, 0.7, 4), multipartite(9, 3)]),
}


@pytest.mark.parametrize("wl", [1, 2])
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_lane_solver_matches_oracle(mce, oracle, name, wl):
    g = GRAPHS[name](mce)
    with mce.DeviceGraph(g) as dg:
        dg.order()
        for level in (1, 2):
            ref = oracle.mce(g, level=level, ipx=True, sub_nodes=True, sub_cliques=True)
            for opts in ({}, {"lane_universe": 16}, {"small_universe": 33}, {"lds_arena_bytes": 1024},
                         {"graph_launch": 1}, {"donate_age_us": 1, "donate_min_p": 4, "donate_check_nodes": 1}):
                print(f"case {name} wl={wl} level={level} {opts}", flush=True)
                res = dg.count(level=level, induced=2, worklist=wl, sub_nodes=True, sub_cliques=True, **opts)
                for k in ("count", "hist", "hash", "tree_nodes"):
                    assert res[k] == ref[k], (k, res[k], ref[k], opts)
                np.testing.assert_array_equal(res["sub_nodes"], ref["sub_nodes"])
                np.testing.assert_array_equal(res["sub_cliques"], ref["sub_cliques"])


@pytest.mark.parametrize("induced", [1, 2])
def test_worker_list_at_its_own_thresholds(mce, oracle, induced):
    # many short launches: every wave must see the end, whoever takes the last task
    g = union(mce, [dense(60, 0.7, 5), dense(90, 0.6, 6)])
    ref = oracle.mce(g, level=1, ipx=induced == 2)
    with mce.DeviceGraph(g) as dg:
        dg.order()
        for i in range(20):
            res = dg.count(level=1, induced=induced, worklist=2)
            for k in ("count", "hist", "hash", "tree_nodes"):
                assert res[k] == ref[k], (i, k)

"""Single-root searches on graphs at the edges of the step launches: one
workgroup or many (64 bitmap words, 2^18 entries), frontiers at the 4,096
vertices a step takes, a workgroup's full list of new vertices, and levels
that go back to the host, against the oracle's levels, schedule and counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def tuples(pairs):
    import graph500_amd
    p = np.asarray(pairs, np.int64)
    t = np.zeros(len(p), graph500_amd.EDGE_DTYPE)
    t["v0_low"], t["v1_low"] = p[:, 0], p[:, 1]
    return t


def check(oracle_mod, edges, roots, mode=2, tuning=None):
    import graph500_amd
    oc = oracle_mod.Csr(edges)
    with graph500_amd.G5Context(0) as c:
        c.edges_append(edges)
        c.construct(mode)
        if tuning:
            c.bfs_set_tuning(**tuning)
        c.prepare_bfs()
        for r in roots:
            print("root", r, flush=True)
            c.run_bfs(r)
            lv, pred, tr = oc.bfs(r)
            assert np.array_equal(c.get_levels(), lv)
            st = c.bfs_stats()
            if mode == 2:
                assert st["direction"] == tr["direction"] and st["nq"] == tr["nq"]
            assert st["reached"] == int((lv != 0xFF).sum())
            assert c.validate()[0]


@pytest.mark.parametrize("rows", [3, 63, 64, 65, 4095, 4096, 4097, 8200])
@pytest.mark.parametrize("mode", [1, 2])
def test_row_counts(oracle_mod, rows, mode):
    rng = np.random.default_rng(rows)
    ring = np.stack([np.arange(rows), (np.arange(rows) + 1) % rows], 1)
    extra = rng.integers(0, rows, (rows * 4, 2))
    check(oracle_mod, tuples(np.concatenate([ring, extra])), [0, rows - 1, rows // 2], mode)


@pytest.mark.parametrize("entries", [(1 << 18) - 2000, (1 << 18) + 2000])
def test_dense_small_graph(oracle_mod, entries):
    rng = np.random.default_rng(7)
    p = rng.integers(0, 2000, (entries // 2, 2))
    check(oracle_mod, tuples(p), [int(p[0, 0]), int(p[5, 1])])


@pytest.mark.parametrize("leaves", [2047, 2049, 4095, 4096, 4097, 9000, 150000])
def test_frontier_sizes(oracle_mod, leaves):
    """A hub with `leaves` children, each with a child of its own, and a tail:
    frontiers of `leaves` vertices top-down and, found by few workgroups, in a
    queue of their own."""
    hub = np.stack([np.zeros(leaves, np.int64), np.arange(1, leaves + 1)], 1)
    kids = np.stack([np.arange(1, leaves + 1), np.arange(leaves + 1, 2 * leaves + 1)], 1)
    tail = np.stack([np.arange(2 * leaves, 2 * leaves + 20), np.arange(2 * leaves + 1, 2 * leaves + 21)], 1)
    check(oracle_mod, tuples(np.concatenate([hub, kids, tail])), [0, 2 * leaves + 20, leaves + 1])


@pytest.mark.parametrize("tuning", [{"small_edges": 0}, {"small_edges": 64}, {"tail_pull": 0}, {"tail_pull": 64}])
def test_tuning(oracle_mod, tuning):
    edges = oracle_mod.generate_edges(15)
    oc = oracle_mod.Csr(edges)
    check(oracle_mod, edges, [int(r) for r in oc.find_roots(6)], 2, tuning)


def test_many_claims_of_few_words(oracle_mod):
    """Rows that all hold the same 200 targets: claims of one word by many
    lanes, across row boundaries too."""
    src = np.repeat(np.arange(1, 3001), 200)
    dst = np.tile(np.arange(4000, 4200), 3000)
    root = np.stack([np.zeros(3000, np.int64), np.arange(1, 3001)], 1)
    check(oracle_mod, tuples(np.concatenate([root, np.stack([src, dst], 1)])), [0, 4100, 17])


@pytest.mark.parametrize("rows", [2047, 2048, 2049, 262143, 262145, 524288, 524289, 1048577])
def test_bottom_up_turns(oracle_mod, rows):
    """Bottom-up levels where one workgroup ends (32 words), where a turn grows
    from one word to two and three (4,096 and 8,192 words) and rows are no
    longer shared out: some hubs, short rows whose first neighbour misses, and
    a path that goes on after them."""
    rng = np.random.default_rng(rows)
    hubs = rng.integers(0, rows // 100, (rows * 2, 1))
    p = np.concatenate([np.concatenate([hubs, rng.integers(0, rows, (rows * 2, 1))], 1),
                        rng.integers(0, rows, (rows, 2)),
                        np.stack([np.arange(rows - 20, rows - 1), np.arange(rows - 19, rows)], 1)])
    check(oracle_mod, tuples(p), [0, rows - 1, int(p[7, 1])])


def test_large_bottom_up_rows(oracle_mod):
    """Bottom-up levels of a graph beyond the steps (over 100,000 bitmap
    words): rows of every length that is searched another way, many of them
    with few reached neighbours."""
    rng = np.random.default_rng(12)
    n = 6_600_000
    ring = np.stack([np.arange(n), rng.integers(0, n, n)], 1)
    lengths = np.concatenate([rng.integers(14, 40, 30000), rng.integers(40, 400, 3000), rng.integers(400, 3000, 60)])
    src = np.repeat(rng.permutation(n)[: len(lengths)], lengths)
    extra = np.stack([src, rng.integers(0, n, len(src))], 1)
    hub = np.stack([np.zeros(9000, np.int64), rng.integers(0, n, 9000)], 1)
    check(oracle_mod, tuples(np.concatenate([ring, extra, hub])), [0, int(src[0]), n - 5])

"""Batch pulls over rows of every length that is searched another way (its
lane alone, a group of 16 lanes, a whole wave after 16 turns), on graphs on
both sides of the sizes where a turn takes 16 rows or 64, against the
oracle's single searches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def build(words, seed):
    """Hubs with rows of chosen lengths over a field of other vertices that
    few searches reach early, in a graph of about 64 * words rows."""
    import graph500_amd
    rng = np.random.default_rng(seed)
    n = 64 * words - 17
    lengths = [1, 2, 8, 9, 10, 16, 17, 18, 25, 33, 257, 258, 400, 401, 450, 1500]
    p = []
    for i, d in enumerate(lengths):
        for c in range(4):
            hub = i * 4 + c
            p.append(np.stack([np.full(d, hub), rng.choice(np.arange(64, n), min(d, n - 64), replace=False)[:d]], 1)
                     if n > 64 + d else np.array([[hub, (hub + 1) % 64]]))
    field = np.arange(64, n)
    p.append(np.stack([field[:-1], field[1:]], 1)[:: 3])
    p.append(rng.integers(64, n, (n // 2, 2)))
    p.append(np.array([[n - 1, 0]]))
    p = np.concatenate(p).astype(np.int64)
    t = np.zeros(len(p), graph500_amd.EDGE_DTYPE)
    t["v0_low"], t["v1_low"] = p[:, 0], p[:, 1]
    return t


@pytest.mark.parametrize("words", [2, 40, 4095, 4098, 12286, 12290])
@pytest.mark.parametrize("mode", [1, 2])
def test_pull_rows(oracle_mod, words, mode):
    import graph500_amd
    edges = build(words, words)
    oc = oracle_mod.Csr(edges)
    ids = np.unique(np.concatenate([edges["v0_low"], edges["v1_low"]]).astype(np.int64))
    rng = np.random.default_rng(3)
    roots = np.concatenate([ids[:8], rng.choice(ids, 29)]).tolist()
    want = {r: oc.bfs(r)[0] for r in set(roots)}
    with graph500_amd.G5Context(0) as c:
        c.edges_append(edges)
        c.construct(mode)
        c.batch_prepare()
        for tuning in ({}, {"lane_rule": 0, "alpha": 1e12, "beta": 0.0}, {"lane_rule": 1, "alpha": 1e12, "beta": 0.0},
                       {"pull_unroll": 4}, {"pull_filter": 1, "pull_unroll": 0}):
            c.batch_set_tuning(**tuning)
            print(words, mode, tuning, flush=True)
            c.run_bfs_batch(roots)
            for lane, r in enumerate(roots):
                assert np.array_equal(c.batch_levels(lane), want[r]), (tuning, lane, r)


@pytest.mark.parametrize("leaves,words", [(8191, 700), (8192, 700), (8193, 700), (30000, 700), (3000, 16384), (3000, 16385)])
def test_level_queue(oracle_mod, leaves, words):
    """Frontiers and bitmaps on both sides of what one workgroup lists beside
    the clears (8,192 vertices, 16,384 words), in pushes, in levels with both
    directions and in the listed pulls at the end of long paths."""
    import graph500_amd
    rng = np.random.default_rng(leaves + words)
    n = 64 * words
    hubs = np.array([0, 1, 2])
    star = np.concatenate([np.stack([np.full(leaves, h), 8 + h * 64 + np.arange(leaves)], 1) for h in hubs])
    field = rng.integers(3, n - 40, (2 * n, 2))
    every = np.stack([np.arange(n - 41), rng.integers(3, n - 41, n - 41)], 1)
    tail = np.stack([np.arange(n - 41, n - 1), np.arange(n - 40, n)], 1)
    p = np.concatenate([star, field, every, tail])
    t = np.zeros(len(p), graph500_amd.EDGE_DTYPE)
    t["v0_low"], t["v1_low"] = p[:, 0], p[:, 1]
    oc = oracle_mod.Csr(t)
    roots = [0, 1, n - 1, int(p[7, 1]), 0, 2, n - 20, 5]
    want = {r: oc.bfs(r)[0] for r in set(roots)}
    with graph500_amd.G5Context(0) as c:
        c.edges_append(t)
        c.construct(2)
        c.batch_prepare()
        for tuning in ({}, {"alpha": 1e-9}, {"alpha": 1.5}, {"mixed_push": 0, "alpha": 64.0}):
            c.batch_set_tuning(**tuning)
            for again in range(2):  # the second batch clears what the first marked
                print(leaves, words, tuning, flush=True)
                c.run_bfs_batch(roots)
                for lane, r in enumerate(roots):
                    assert np.array_equal(c.batch_levels(lane), want[r]), (tuning, lane, r)

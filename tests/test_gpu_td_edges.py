"""Top-down levels whose edge count the level before has summed: a frontier of
more than 4,096 vertices on both sides of 2^20 edges, from one such frontier
to the next."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, B, PAIRS = 5000, 6000, 6_100_000


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("leaves", [1, 100, 172, 173, 200])
def test_counted_levels(leaves, mode):
    """root - A - B - leaves, beside pairs that keep the frontiers below a
    2000th of the vertices; B's rows hold 6,000 (leaves + 1) + 4,000 edges."""
    import graph500_amd
    print("leaves", leaves, "mode", mode, flush=True)
    a = 1 + np.arange(A)
    b = 1 + A + np.arange(B)
    leaf = 1 + A + B + np.arange(B * leaves)
    pair = 1 + A + B + B * leaves + np.arange(2 * PAIRS)
    links = 10000
    src = np.concatenate([np.zeros(A, np.int64), a[np.arange(links) % A], b[np.arange(B * leaves) % B], pair[::2]])
    dst = np.concatenate([a, b[np.arange(links) % B], leaf, pair[1::2]])
    t = np.zeros(len(src), graph500_amd.EDGE_DTYPE)
    t["v0_low"], t["v1_low"] = src, dst
    want = np.full(1 << 24, 0xFF, np.uint8)
    want[0], want[a], want[b], want[leaf] = 0, 1, 2, 3
    with graph500_amd.G5Context(0) as ctx:
        ctx.edges_append(t)
        ctx.construct(mode, release_edges=True)
        ctx.prepare_bfs()
        for _ in range(2):
            ctx.run_bfs(0)
            st = ctx.bfs_stats()
            assert st["nq"][:3] == [A, B, B * leaves] and st["direction"][:3] == [1, 1, 1]
            assert np.array_equal(ctx.get_levels(), want)
            ok, errors = ctx.validate()
            assert ok, errors
            assert ctx.teps_edges() == A + links + B * leaves

"""Which levels of a batch pull, on both sides of the size from which a root
that is over its own threshold waits for the union of the frontiers for good;
levels against the oracle either way."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PULL, PUSH = 0, 1


def grid(n, w):
    i = np.arange(n * w)
    x, y = i % n, i // n
    return (np.concatenate([i[x < n - 1], i[y < w - 1]]),
            np.concatenate([i[x < n - 1] + 1, i[y < w - 1] + n]))


def run(ctx, oc, roots):
    ctx.batch_prepare()
    ctx.run_bfs_batch(roots)
    for lane, r in enumerate(roots):
        assert np.array_equal(ctx.batch_levels(lane), oc.bfs(int(r), want_pred=False)[0])
    return ctx.batch_stats()["direction"]


@pytest.mark.parametrize("n,w", [(200, 1), (120, 4), (200, 4)])
@pytest.mark.parametrize("nroots", [2, 8])
def test_long_small_graphs_pull(oracle_mod, n, w, nroots):
    """A frontier of a few vertices of a small graph: a root waits one level
    for the union, pulls, and keeps pulling."""
    import graph500_amd
    print("grid", n, w, nroots, flush=True)
    a, b = grid(n, w)
    t = np.zeros(len(a), graph500_amd.EDGE_DTYPE)
    t["v0_low"], t["v1_low"] = a, b
    with graph500_amd.G5Context(0) as ctx:
        ctx.edges_append(t)
        ctx.construct(2)
        d = run(ctx, oracle_mod.Csr(t), ctx.find_roots(nroots))
        assert len(d) > 60
        assert d.count(PULL) >= len(d) - 8


@pytest.mark.parametrize("w,large", [(1024, False), (8192, True)])
def test_large_graphs_wait(oracle_mod, w, large):
    """Two roots in a grid with chords, 110 to 145 levels: the small graph
    pulls for them most of the time, the large one pushes."""
    import graph500_amd
    print("chords", w, flush=True)
    a, b = grid(128, w)
    i = np.arange(128 * w)
    at = i[i // 128 % 16 == 0]
    rng = np.random.default_rng(3)
    a = np.concatenate([a, at])
    b = np.concatenate([b, (at + 128 * 16 * rng.integers(0, w // 16, len(at))) % (128 * w)])
    t = np.zeros(len(a), graph500_amd.EDGE_DTYPE)
    t["v0_low"], t["v1_low"] = a, b
    with graph500_amd.G5Context(0) as ctx:
        ctx.edges_append(t)
        ctx.construct(2)
        assert (ctx.graph_info()["nnz"] >= 1 << 22) == large
        d = run(ctx, oracle_mod.Csr(t), ctx.find_roots(2, 7, 3))
        assert len(d) > 90
        assert d.count(PUSH) > 0.8 * len(d) if large else d.count(PUSH) < 0.4 * len(d)


@pytest.mark.parametrize("scale", [14, 16, 19])
def test_growing_graphs_wait_one_level(oracle_mod, scale):
    """8 roots of a Kronecker graph, of which some are over their own threshold
    at level 2 where the union of all is below its own, and no longer at level
    3: all push at level 2, no mixed level."""
    import graph500_amd
    print("scale", scale, flush=True)
    with graph500_amd.G5Context(0) as ctx:
        ctx.generate_kronecker(scale, 16, 2, 3)
        t = ctx.edges_download()
        ctx.construct(2)
        d = run(ctx, oracle_mod.Csr(t), ctx.find_roots(4 if scale == 16 else 8, 7, 3))
        assert d[:3] == [PUSH, PUSH, PULL]

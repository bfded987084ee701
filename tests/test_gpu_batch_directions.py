"""Which levels of a batch pull, on both sides of the size from which the
union of the frontiers decides with each root's own frontier; levels against
the oracle either way."""
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
    """A frontier of a few vertices of a small graph: once a root pulls it
    keeps pulling, as its own frontier says."""
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


@pytest.mark.parametrize("scale,mixed", [(16, True), (19, False)])
def test_union_decides_on_large_graphs(oracle_mod, scale, mixed):
    """8 roots, of which some are over their own threshold at level 2 where
    the union of all is below its own: the small graph pulls for them, the
    large one pushes for all."""
    import graph500_amd
    print("scale", scale, flush=True)
    with graph500_amd.G5Context(0) as ctx:
        ctx.generate_kronecker(scale, 16, 5, 9)
        t = ctx.edges_download()
        ctx.construct(2)
        assert (ctx.graph_info()["nnz"] < 1 << 22) == mixed
        d = run(ctx, oracle_mod.Csr(t), ctx.find_roots(8, 7, 3))
        assert d[0] == PUSH and (d[1] == PUSH) != mixed

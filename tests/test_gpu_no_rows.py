"""Searches of a graph whose tuples are all self loops: in reorder modes 1 and
2 it has no row at all.  Every root is the whole tree of its search; mode 0
keeps a row per id, so only there does the root's own weight (its loops) count
as traversed edges."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LOOPS = [3, 3, 5, 6]
N = 8


@pytest.fixture(params=[0, 1, 2])
def graph(request):
    import graph500_amd
    print("loops only, mode", request.param, flush=True)
    t = np.zeros(len(LOOPS), graph500_amd.EDGE_DTYPE)
    t["v0_low"] = t["v1_low"] = LOOPS
    with graph500_amd.G5Context(0) as c:
        c.edges_append(t)
        c.construct(request.param)
        yield c, request.param


def levels_of(root):
    lv = np.full(N, 0xFF, np.uint8)
    lv[root] = 0
    return lv


def edges_of(root, mode):
    return LOOPS.count(root) if mode == 0 else 0


def test_search(graph):
    ctx, mode = graph
    ctx.prepare_bfs()
    for root in (3, 5, 0, 7):
        print("root", root, flush=True)
        ctx.run_bfs(root)
        assert np.array_equal(ctx.get_levels(), levels_of(root))
        pred = ctx.get_pred()
        assert pred[root] == root and (np.delete(pred, root) == -1).all()
        assert ctx.teps_edges() == edges_of(root, mode)
        ok, errors = ctx.validate()
        assert ok, errors
        for check in (ctx.validate_pred, ctx.validate_pred_noalloc):
            ok, errors, edges = check(root, pred)
            assert ok and edges == edges_of(root, mode), errors
        st = ctx.bfs_stats()
        assert st["num_levels"] == 2 and st["nq"] == [0] and st["reached"] == 1


def test_batch(graph):
    ctx, mode = graph
    roots = [3, 5, 0, 7, 3]
    ctx.batch_prepare()
    ctx.run_bfs_batch(roots)
    assert list(ctx.batch_teps_edges()) == [edges_of(r, mode) for r in roots]
    for lane, root in enumerate(roots):
        assert np.array_equal(ctx.batch_levels(lane), levels_of(root))


@pytest.mark.parametrize("solo", [0, 4])
def test_server(graph, solo):
    import graph500_amd
    ctx, mode = graph
    if mode == 0:
        return  # the server takes graphs built with mode 1 or 2
    roots = [3, 5, 0, 7, 3]
    q = np.zeros(len(roots), graph500_amd.QUERY_DTYPE)
    q["root"], q["keep"] = roots, [1, 1, 0, 1, 0]
    with graph500_amd.G5Server([ctx], answer_buffers=4, solo=solo, solo_slots=2) as srv:
        res, _ = srv.run(q)
        assert (res["edges"] == 0).all()
        for i in np.flatnonzero(q["keep"]):
            assert np.array_equal(srv.levels(res["request"][i], N), levels_of(roots[i]))

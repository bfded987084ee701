"""The time of a search is a time for every root: also for one without edges,
whose search ends before its first level."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [9, 14])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_device_time_of_a_root_without_edges(scale, mode):
    import graph500_amd
    print("scale", scale, "mode", mode, flush=True)
    with graph500_amd.G5Context(0) as ctx:
        ctx.generate_kronecker(scale, 16)
        ctx.construct(mode)
        alone = next(v for v in range(1 << scale) if not ctx.has_edge(v))
        ctx.prepare_bfs()
        for root in (alone, int(ctx.find_roots(1)[0]), alone):
            ctx.run_bfs(root)
            st = ctx.bfs_stats()
            assert 0 < st["device_ms"] < 1000
            if root == alone:
                assert st["num_levels"] == 2 and st["direction"] == [1] and st["nq"] == [0] and st["reached"] == 1
                lv = ctx.get_levels()
                assert lv[root] == 0 and (lv == 0xFF).sum() == len(lv) - 1
            else:
                assert st["reached"] > 1 and len(st["nq"]) == st["num_levels"] - 1

"""A construction beside other users of the device: two 8-byte keys per
directed entry and the arrays per id are its peak, so it runs where that much
is free; the columns are allocated after the first of the two has gone back."""
import pytest

pytestmark = pytest.mark.gpu


def test_peak_is_two_key_arrays():
    import torch

    import graph500_amd
    scale, ef = 24, 16
    m, n = ef << scale, 1 << scale
    with graph500_amd.G5Context(0) as ctx:
        ctx.generate_kronecker(scale, ef)
        # two key arrays and 48 bytes an id (27 are needed), of which the tuples hold 12 m now;
        # the columns (about 8 m bytes) do not fit beside the keys
        leave = 32 * m + 48 * n - 12 * m
        free, _ = torch.cuda.mem_get_info(0)
        print("free", free, "leave", leave, flush=True)
        held = [torch.empty((free - leave) // 8, dtype=torch.uint8, device="cuda:0") for _ in range(8)]
        print("held", sum(t.numel() for t in held), "free", torch.cuda.mem_get_info(0)[0], flush=True)
        try:
            ctx.construct(2, release_edges=True)
            info = ctx.graph_info()
        finally:
            del held
            torch.cuda.empty_cache()
        assert info["num_verts"] == n and info["directed_before"] == 2 * (m - info["num_self_loops"])
        # the graph the same tuples give without that
        ctx.generate_kronecker(scale, ef)
        ctx.construct(2, release_edges=True)
        other = ctx.graph_info()
        for key in ("nnz", "num_active", "max_degree", "num_self_loops", "max_used_vertex"):
            assert info[key] == other[key]

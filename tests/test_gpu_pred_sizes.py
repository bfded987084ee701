"""Predecessors into pinned memory on both sides of the size (16 MiB) up to
which the kernel stores them itself: the same as into ordinary memory, and
nothing beyond the last."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [20, 21, 22])
def test_pinned_equals_ordinary(scale):
    import graph500_amd
    print("scale", scale, flush=True)
    with graph500_amd.G5Context(0) as ctx:
        ctx.generate_kronecker(scale, 8)
        ctx.construct(2)
        n, root = ctx.pred_size(), int(ctx.find_roots(1)[0])
        path = next(x.split()[-1] for x in open("/proc/self/maps") if "libamdhip64" in x)
        hip, p = ctypes.CDLL(path), ctypes.c_void_p()
        size = (n + 4) * 8
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(size), 0) == 0
        try:
            pinned = np.frombuffer((ctypes.c_char * size).from_address(p.value), np.int64)
            pinned[:] = -7
            ctx.prepare_bfs()
            ctx.run_bfs(root)
            ctx.get_pred(pinned[:n])
            pred = ctx.get_pred()
            assert np.array_equal(pinned[:n], pred) and (pinned[n:] == -7).all()
            ok, errors, edges = ctx.validate_pred(root, pred)
            assert ok and edges == ctx.teps_edges(), errors
        finally:
            hip.hipHostFree(p)

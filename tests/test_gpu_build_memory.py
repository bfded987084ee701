"""A construction beside other users of the device: two 8-byte keys per
directed entry and the arrays per id are its peak, so it runs where that much
is free; the columns are allocated after the first of the two has gone back."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def hip():
    """The HIP runtime that the library uses."""
    import graph500_amd
    graph500_amd.G5Context(0).close()
    path = next(x.split()[-1] for x in open("/proc/self/maps") if "libamdhip64" in x)
    return ctypes.CDLL(path)


def free_bytes(hip):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_peak_is_two_key_arrays(hip):
    import graph500_amd
    scale, ef = 24, 16
    m, n = ef << scale, 1 << scale
    held = []
    with graph500_amd.G5Context(0) as ctx:
        ctx.generate_kronecker(scale, ef)
        # two key arrays and 48 bytes an id (27 are needed), of which the tuples hold 12 m now;
        # the columns (about 8 m bytes) do not fit beside the keys
        leave = 32 * m + 48 * n - 12 * m
        try:
            # in pieces, to within 1.5 GB (the unfreed key array would need 2.1 more than there is)
            while (left := free_bytes(hip) - leave) > 3 << 29:
                p = ctypes.c_void_p()
                if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(max(1 << 30, left // 4))) != 0:
                    pytest.skip("the device's free memory cannot be had in pieces")
                held.append(p)
            print("held in", len(held), "free", free_bytes(hip), flush=True)
            assert left >= 0
            ctx.construct(2, release_edges=True)
            info = ctx.graph_info()
        finally:
            for p in held:
                hip.hipFree(p)
        assert info["num_verts"] == n and info["directed_before"] == 2 * (m - info["num_self_loops"])
        # the graph the same tuples give without that
        ctx.generate_kronecker(scale, ef)
        ctx.construct(2, release_edges=True)
        other = ctx.graph_info()
        for key in ("nnz", "num_active", "max_degree", "num_self_loops", "max_used_vertex"):
            assert info[key] == other[key]

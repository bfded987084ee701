"""Answers on their way to the host: pinned, misaligned and ordinary buffers
on both sides of the sizes where the way changes (256 KiB, 2^19 rows, the
levels a launch's arguments hold), against the oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def graph(n_bits, pairs, tail):
    """`pairs` random edges among the first half of the ids, then a path."""
    import graph500_amd
    rng = np.random.default_rng(n_bits)
    n = 1 << n_bits
    p = rng.integers(0, max(n - tail - 1, 1), (pairs, 2))
    p = p[p[:, 0] != p[:, 1]]
    path = np.arange(n - tail - 1, n) if tail else np.array([n - 2, n - 1])
    p = np.concatenate([p, np.stack([path[:-1], path[1:]], 1), [[0, path[0]]]])
    t = np.zeros(len(p), graph500_amd.EDGE_DTYPE)
    t["v0_low"], t["v1_low"] = p[:, 0], p[:, 1]
    return t


@pytest.fixture
def pinned():
    """Pinned host memory from the HIP runtime that the library uses."""
    import graph500_amd
    graph500_amd.G5Context(0).close()
    path = next(x.split()[-1] for x in open("/proc/self/maps") if "libamdhip64" in x)
    hip, held = ctypes.CDLL(path), []

    def alloc(count, dtype):
        p = ctypes.c_void_p()
        size = count * np.dtype(dtype).itemsize
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(size), 0) == 0
        held.append(p)
        return np.frombuffer((ctypes.c_char * size).from_address(p.value), dtype)

    yield alloc
    for p in held:
        hip.hipHostFree(p)


def buffers(pinned, n, dtype):
    held = pinned(n + 16, dtype)
    yield "pinned", held[:n]
    yield "pinned+1", held[1:n + 1]
    yield "ordinary", np.empty(n, dtype)
    yield "ordinary+1", np.empty(n + 1, dtype)[1:]


@pytest.mark.parametrize("n_bits,pairs,tail", [(2, 3, 1), (3, 12, 0), (4, 30, 4), (5, 90, 28), (12, 9000, 23), (12, 9000, 24),
                                               (15, 90000, 40), (18, 800000, 2), (19, 3000000, 3), (20, 9000000, 40)])
def test_answers_to_any_buffer(oracle_mod, pinned, n_bits, pairs, tail):
    import graph500_amd
    edges = graph(n_bits, pairs, tail)
    n = 1 << n_bits
    oc = oracle_mod.Csr(edges)
    roots = [int(edges["v0_low"][0]), n - 1, n - 2]
    want = [oc.bfs(r)[0] for r in roots]
    degree = np.bincount(np.concatenate([edges["v0_low"], edges["v1_low"]]).astype(np.int64), minlength=n)
    with graph500_amd.G5Context(0) as c:
        c.edges_append(edges)
        c.construct(2)
        c.prepare_bfs()
        c.batch_prepare()
        c.run_bfs_batch(roots)
        for lane, w in enumerate(want):
            for name, buf in buffers(pinned, n, np.uint8):
                buf[:] = 77
                assert np.array_equal(c.batch_levels(lane, buf), w), (lane, name)
        many = c.batch_teps_edges()
        assert np.array_equal(many, c.batch_teps_edges())
        for r, w, e in zip(roots, want, many):
            c.run_bfs(r)
            for name, buf in buffers(pinned, n, np.uint8):
                buf[:] = 77
                assert np.array_equal(c.get_levels(buf), w), (r, name)
            for name, buf in buffers(pinned, n, np.int64):
                buf[:] = -77
                c.get_pred(buf)
                assert np.array_equal(buf >= 0, w != 0xFF) and buf[r] == r, (r, name)
            assert c.teps_edges() == e == int(degree[w != 0xFF].sum()) // 2

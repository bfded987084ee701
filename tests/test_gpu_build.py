"""CSR construction on the GPU against a plain numpy build of the same rows,
at the sizes where its partition and sort passes change shape: partial and
whole tiles (3,072 tuples), one and several id ranges, sub-buckets of 2,048
positions, both relabelling forms, rows that cross sub-buckets, and the inputs
that leave the LDS sort for the radix sort (thousands of copies of one tuple, a
row of more than 2^24 entries)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def tuples(a, b):
    import graph500_amd
    t = np.zeros(len(a), graph500_amd.EDGE_DTYPE)
    t["v0_low"], t["v1_low"] = a, b
    return t


def reference(a, b, mode):
    """offsets, cols, new2old, weight as the construction defines them."""
    a, b = a.astype(np.int64), b.astype(np.int64)
    n = 1 << int(np.bitwise_or.reduce(a | b)).bit_length()
    keep = a != b
    deg = np.bincount(a[keep], minlength=n) + np.bincount(b[keep], minlength=n)
    loops = np.bincount(a[~keep], minlength=n)
    if mode == 2:
        new2old = np.argsort(-deg, kind="stable")
    elif mode == 1:
        new2old = np.argsort(deg == 0, kind="stable")
    else:
        new2old = np.arange(n)
    old2new = np.empty(n, np.int64)
    old2new[new2old] = np.arange(n)
    rows = n if mode == 0 else int((deg > 0).sum())
    na, nb = old2new[a[keep]], old2new[b[keep]]
    keys = np.unique(np.concatenate([(na << 32) | nb, (nb << 32) | na]))
    offsets = np.searchsorted(keys >> 32, np.arange(rows + 1))
    return offsets, keys & 0xFFFFFFFF, new2old, (deg + 2 * loops)[new2old[:rows]]


def check(ctx, a, b, mode, case):
    print(case, "mode", mode, len(a), flush=True)
    ctx.edges_release()
    ctx.edges_append(tuples(a, b))
    ctx.construct(mode, release_edges=True)
    g = ctx.graph_download()
    off, cols, new2old, weight = reference(a, b, mode)
    assert np.array_equal(g["new2old"], new2old)
    assert np.array_equal(g["offsets"], off)
    assert np.array_equal(g["cols"], cols)
    assert np.array_equal(g["weight"], weight)


@pytest.fixture(scope="module")
def ctx():
    import graph500_amd
    c = graph500_amd.G5Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("scale,m", [(1, 1), (3, 5), (6, 700), (7, 3071), (9, 3072), (13, 3073), (14, 100001),
                                     (17, 262144), (20, 500000), (21, 500000), (24, 300007), (26, 50021)])
def test_rows_equal_numpy(ctx, scale, m, mode):
    rng = np.random.default_rng(scale * 3 + mode)
    n = 1 << scale
    # half the endpoints on a few hubs, the rest anywhere; the top id present
    a = np.where(rng.random(m) < 0.5, rng.integers(0, n, m), (rng.pareto(1.0, m) * 3).astype(np.int64) * 7919 % n)
    b = rng.integers(0, n, m)
    a[0], b[0] = n - 1, 0
    check(ctx, a, b, mode, "scale %d" % scale)


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("copies", [4095, 4097, 20000])
def test_many_copies_of_one_tuple(ctx, copies, mode):
    rng = np.random.default_rng(copies)
    a, b = rng.integers(0, 1 << 12, 50000), rng.integers(0, 1 << 12, 50000)
    a[:copies], b[:copies] = 5, 4000
    check(ctx, a, b, mode, "copies %d" % copies)


@pytest.mark.parametrize("scale", [25, 26, 27])
def test_degrees_of_wide_ranges(ctx, scale):
    """One, two and four workgroups count a range of ids; ranges of entries
    below, at and beyond a workgroup's batch (8,192), from odd places on."""
    rng = np.random.default_rng(scale)
    n, width = 1 << scale, 1 << (scale - 10)
    sizes = [1, 8190, 8191, 8192, 8193, 16385, 3, 24575, 40001]
    a = np.concatenate([rng.integers(k * 7 * width, (k * 7 + 1) * width, size) for k, size in enumerate(sizes)])
    a = np.append(a, [n - 1, 70 * width, 71 * width - 1])
    b = rng.integers(100 * width, n, len(a))
    check(ctx, a, b, 1, "wide %d" % scale)


@pytest.mark.parametrize("mode", [0, 2])
def test_only_loops_and_loops_between(ctx, mode):
    a = np.array([3, 3, 5], np.int64)
    check(ctx, a, a, mode, "loops only")
    rng = np.random.default_rng(9)
    a, b = rng.integers(0, 4096, 9001), rng.integers(0, 4096, 9001)
    b[::3] = a[::3]
    check(ctx, a, b, mode, "a third loops")


@pytest.mark.parametrize("leaves", [300000, (1 << 24) + 4099])
def test_star(ctx, leaves):
    print("star", leaves, flush=True)
    ctx.edges_release()
    leaf = np.arange(1, leaves + 1, dtype=np.int64)
    ctx.edges_append(tuples(np.zeros(leaves, np.int64), leaf))
    ctx.construct(2, release_edges=True)
    g = ctx.graph_download()
    assert np.array_equal(g["cols"][:leaves], leaf)
    assert not g["cols"][leaves:].any() and len(g["cols"]) == 2 * leaves
    assert np.array_equal(g["offsets"], np.concatenate([[0], np.arange(leaves, 2 * leaves + 1)]))


@pytest.mark.parametrize("scale,edgefactor", [(19, 13), (20, 17), (33, 1)])
def test_generator_slices(oracle_mod, scale, edgefactor):
    """Runs that do not fill the last workgroup, and ids beyond 32 bits."""
    import graph500_amd
    print("slices", scale, edgefactor, flush=True)
    m = edgefactor << scale
    with graph500_amd.G5Context(0) as c:
        c.generate_kronecker(scale, edgefactor, 5, 9)
        for start in (0, 255, m // 3, (1 << min(scale, 32)) - 300, m - 1001):
            got = c.edges_download(start, 1001 if start + 1001 <= m else m - start)
            exp = oracle_mod.generate_edges(scale, edgefactor, 5, 9, start=start, end=start + len(got))
            assert np.array_equal(got, exp), start


@pytest.mark.parametrize("scale", [1, 2, 3, 4, 5, 6, 9, 10, 11])
@pytest.mark.parametrize("a,bc", [(5700, 1900), (5500, 100), (10000, 0), (0, 5000), (0, 0), (1, 4999), (9998, 1)])
def test_generator_parameters(oracle_mod, scale, a, bc):
    """Levels in fives and the rest, and thresholds at the ends of their range."""
    import graph500_amd
    with graph500_amd.G5Context(0) as c:
        c.generate_kronecker(scale, 23, 7, 11, a, bc)
        got = c.edges_download()
        assert np.array_equal(got, oracle_mod.generate_edges(scale, 23, 7, 11, a, bc)), (scale, a, bc)

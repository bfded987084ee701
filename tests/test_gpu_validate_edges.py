"""The validator's count of edges that break the level rule, against a count
over every entry of the downloaded rows: graphs of a few entries, of short
rows only, of one row that many runs of entries share, with empty rows, and
with more rows than the ones whose levels are kept in LDS."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def build(kind):
    import graph500_amd
    rng = np.random.default_rng(5)
    if kind == "pair":
        p = [(0, 1)]
    elif kind == "path":
        p = [(i, i + 1) for i in range(300)]
    elif kind == "ring":
        i = np.arange(150000)
        p = np.stack([i, (i + 1) % len(i)], 1)
    elif kind == "star":
        i = np.arange(1, 400000)
        p = np.stack([np.where(i % 3, 0, 399999), i], 1)
    elif kind == "clique":
        p = [(i, j) for i in range(257) for j in range(i)]
    elif kind == "holes":
        p = np.concatenate([rng.integers(0, 1000, (5000, 2)) * 97, [(0, 97 * 999)]])
    else:
        p = None
    c = graph500_amd.G5Context(0)
    if p is None:
        c.generate_kronecker(kind, 16, 3, 4)
    else:
        p = np.asarray(p, np.int64)
        t = np.zeros(len(p), graph500_amd.EDGE_DTYPE)
        t["v0_low"], t["v1_low"] = p[:, 0], p[:, 1]
        c.edges_append(t)
    return c


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("kind", ["pair", "path", "ring", "star", "clique", "holes", 9, 13, 16, 19])
def test_level_rule_counts(kind, mode):
    with build(kind) as c:
        c.construct(mode)
        c.prepare_bfs()
        g = c.graph_download()
        rows = len(g["offsets"]) - 1
        old = g["new2old"][:rows].astype(np.int64)
        src = np.repeat(np.arange(rows), np.diff(g["offsets"].astype(np.int64)))
        dst = g["cols"].astype(np.int64)
        root = int(c.find_roots(1)[0])
        rng = np.random.default_rng(11)
        n = c.pred_size()
        if kind not in ("path", "ring"):  # deeper than a search goes
            c.run_bfs(root)
            pred = c.get_pred()
        else:
            pred = np.full(n, -1, np.int64)
            pred[root] = root
        for planted in (0, 1, 5, rows // 3):
            p = pred.copy()
            v = old[rng.integers(0, rows, planted)] if planted else np.zeros(0, np.int64)
            p[v] = np.where(rng.random(len(v)) < 0.3, -1, (v & ((1 << 48) - 1)) | (rng.integers(0, 9, len(v)) << 48))
            lv = np.where(p == -1, -100, p >> 48)[old]
            a, b = lv[src], lv[dst]
            want = int((((a < 0) != (b < 0)) | ((a >= 0) & (b >= 0) & (np.abs(a - b) > 1))).sum())
            ok, err, edges = c.validate_pred(root, p)
            print(kind, mode, planted, rows, want, err, flush=True)
            assert err["edge"] == want
            assert edges == int(g["weight"][lv >= 0].astype(np.int64).sum()) // 2

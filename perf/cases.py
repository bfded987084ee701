"""The work that programs have this library do, as cases to be timed.

A case is one of five kinds, each a pass through the public Python API:

  search    run_bfs from each of the case's roots on a resident graph, with
            the levels of every root (out="all") or, on graphs whose level
            arrays a benchmark does not keep, each root's traversed-edge
            count and the last root's levels (out="edges")
  batch     run_bfs_batch over up to 64 roots, the traversed edges of every
            root, and the level arrays of the first `lanes` roots
  build     a graph from nothing (generator, or tuples in host memory) to
            the answer of its first search: tuples, CSR, root, BFS
  validate  the benchmark's step for one root: search, fetch the
            predecessors, validate them, keep the levels
  serve     a burst of queries over several resident graphs through a
            G5Server, some answers kept and fetched

Parents are not returned anywhere: several are valid and a search may pick
any.  Everything returned is a whole number that the graph and root fix.
"""
import random

import numpy as np
import torch

import graph500_amd as g5


def listed():
    return [
        # one query on a tiny graph: what a unit test or a small tool does; launches and host latency only
        {"name": "search_s10", "kind": "search", "scale": 10, "edgefactor": 16, "mode": 2, "roots": 1, "out": "all"},
        # one query on the smoke-test graph, the latency of a single small answer
        {"name": "search_s16", "kind": "search", "scale": 16, "edgefactor": 16, "mode": 2, "roots": 1, "out": "all"},
        # a few queries on a mid-size graph, every answer fetched
        {"name": "search_s21", "kind": "search", "scale": 21, "edgefactor": 16, "mode": 2, "roots": 4, "out": "all"},
        # the Graph500 loop at the benchmark's own size: search after search, the edge count of each
        {"name": "search_s28", "kind": "search", "scale": 28, "edgefactor": 16, "mode": 2, "roots": 8, "out": "edges"},
        # 64 answers on a small graph in one batch, all fetched
        {"name": "batch_s12", "kind": "batch", "scale": 12, "edgefactor": 16, "mode": 2, "roots": 64, "lanes": 16},
        # a batch that is not full, all answers fetched
        {"name": "batch_s19_odd", "kind": "batch", "scale": 19, "edgefactor": 16, "mode": 2, "roots": 37, "lanes": 37},
        # the batched throughput benchmark, levels of a few roots fetched to be checked
        {"name": "batch_s26", "kind": "batch", "scale": 26, "edgefactor": 16, "mode": 2, "roots": 64, "lanes": 4},
        # a small spec-2012 graph (tree tuples first, odd edge factor), as the tests build them
        {"name": "build_s13_2012", "kind": "build", "scale": 13, "edgefactor": 7, "mode": 2, "source": "spec2012",
         "drop": 0},
        # a caller's own ragged edge list handed over from host memory, vertices in input order first (mode 1)
        {"name": "build_s18_host", "kind": "build", "scale": 18, "edgefactor": 16, "mode": 1, "source": "host",
         "drop": 4097},
        # kernel 1 of the benchmark at a size where the sort carries the time
        {"name": "build_s25", "kind": "build", "scale": 25, "edgefactor": 16, "mode": 2, "source": "kronecker",
         "drop": 0},
        # the benchmark's whole step for one root: search, predecessors, validation
        {"name": "validate_s21", "kind": "validate", "scale": 21, "edgefactor": 16, "mode": 2},
        # a burst over a mix of resident graphs, more queries than the single-root slots take
        {"name": "serve_mix", "kind": "serve", "scales": "17,20,22", "edgefactor": 16, "queries": 160, "keep": 6},
    ]


def draw(rng):
    kind = rng.choice(["search", "search", "batch", "batch", "build", "build", "validate", "serve"])
    ef = rng.choice([16, 16, 16, rng.randint(4, 31)])
    mode = rng.choice([2, 2, 2, 1, 0])
    if kind == "search":
        return {"kind": kind, "scale": rng.randint(8, 25), "edgefactor": ef, "mode": mode,
                "roots": rng.randint(1, 5), "out": rng.choice(["all", "edges"])}
    if kind == "batch":
        roots = rng.randint(2, 64)
        return {"kind": kind, "scale": rng.randint(8, 24), "edgefactor": ef, "mode": max(mode, 1), "roots": roots,
                "lanes": rng.randint(1, min(roots, 8))}
    if kind == "build":
        source = rng.choice(["kronecker", "kronecker", "spec2012", "host"])
        scale = rng.randint(8, 19 if source == "host" else 23)
        return {"kind": kind, "scale": scale, "edgefactor": ef, "mode": mode, "source": source,
                "drop": rng.randint(1, 1 << (scale - 1)) if source == "host" else 0}
    if kind == "validate":
        return {"kind": kind, "scale": rng.randint(8, 22), "edgefactor": ef, "mode": mode}
    scales = sorted(rng.sample(range(12, 22), rng.randint(2, 3)))
    return {"kind": kind, "scales": ",".join(map(str, scales)), "edgefactor": ef, "queries": rng.randint(20, 150),
            "keep": rng.randint(1, 6)}


def _graph(scale, ef, mode, rng, source="kronecker"):
    ctx = g5.G5Context(0)
    gen = ctx.generate_graph_spec2012 if source == "spec2012" else ctx.generate_kronecker
    gen(scale, ef, rng.getrandbits(40), rng.getrandbits(40))
    ctx.construct(mode, release_edges=True)
    return ctx


def _host(shape, dtype):
    """A host buffer that the program keeps for what it fetches: pinned."""
    return torch.empty(shape, dtype=dtype, pin_memory=True).numpy()


def prepare(case, seed):
    rng = random.Random(seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "build":
        n, ef = 1 << case["scale"], case["edgefactor"]
        st["seeds"] = (rng.getrandbits(40), rng.getrandbits(40))
        st["ctx"] = ctx = g5.G5Context(0)
        st["out"] = _host(n, torch.uint8)
        if case["source"] == "host":
            ctx.generate_kronecker(case["scale"], ef, *st["seeds"])
            st["tuples"] = ctx.edges_download(0, n * ef - case["drop"])
            ctx.edges_release()
        return st
    if kind == "serve":
        ctxs = [_graph(int(s), case["edgefactor"], 2, rng) for s in case["scales"].split(",")]
        st["server"] = g5.G5Server(ctxs, answer_buffers=128, solo=8, solo_slots=3)
        roots = [c.find_roots(64, rng.getrandbits(30), 3) for c in ctxs]
        q = np.zeros(case["queries"], g5.QUERY_DTYPE)
        # the kept answers come from the graphs in turn, of the other queries half go to the middle
        # graph and the rest evenly; a query every 10 us
        for i in range(len(q)):
            keep = i < case["keep"]
            g = i % len(ctxs) if keep else len(ctxs) // 2 if rng.random() < 0.5 else rng.randrange(len(ctxs))
            q[i] = (g, int(keep), int(rng.choice(roots[g].tolist())), i * 1e-5)
        st["queries"] = q
        st["sizes"] = [c.pred_size() for c in ctxs]
        return st
    ctx = _graph(case["scale"], case["edgefactor"], case["mode"], rng)
    n = ctx.pred_size()
    st["ctx"] = ctx
    st["roots"] = [int(r) for r in ctx.find_roots(case.get("roots", 1), rng.getrandbits(30), 3)]
    if kind == "batch":
        ctx.batch_prepare()
        st["out"] = _host((min(case["lanes"], len(st["roots"])), n), torch.uint8)
    else:
        ctx.prepare_bfs()
        st["out"] = _host((len(st["roots"]) if case.get("out") == "all" else 1, n), torch.uint8)
    if kind == "validate":
        st["pred"] = _host(n, torch.int64)
    return st


def _run_search(st):
    ctx, out = st["ctx"], st["out"]
    if st["case"]["out"] == "all":
        for i, r in enumerate(st["roots"]):
            ctx.run_bfs(r)
            ctx.get_levels(out[i])
        return {"levels": out}
    edges = []
    for r in st["roots"]:
        ctx.run_bfs(r)
        edges.append(ctx.teps_edges())
    ctx.get_levels(out[0])
    return {"edges": np.array(edges, np.int64), "levels": out}


def _run_batch(st):
    ctx, out = st["ctx"], st["out"]
    ctx.run_bfs_batch(st["roots"])
    edges = ctx.batch_teps_edges()
    for lane in range(len(out)):
        ctx.batch_levels(lane, out[lane])
    return {"edges": edges, "levels": out}


def _run_build(st):
    ctx, case = st["ctx"], st["case"]
    if case["source"] == "host":
        tuples, chunk = st["tuples"], 1 << 23  # the edge list comes in chunks of 8 Mi tuples
        for i in range(0, len(tuples), chunk):
            ctx.edges_append(tuples[i : i + chunk])
    elif case["source"] == "spec2012":
        ctx.generate_graph_spec2012(case["scale"], case["edgefactor"], *st["seeds"])
    else:
        ctx.generate_kronecker(case["scale"], case["edgefactor"], *st["seeds"])
    ctx.construct(case["mode"], release_edges=True)
    root = int(ctx.find_roots(1)[0])
    ctx.prepare_bfs()
    ctx.run_bfs(root)
    info = ctx.graph_info()
    # a caller's list may leave the top ids unused: the answer has the graph's own size
    levels = ctx.get_levels(st["out"][: info["num_verts"]])
    return {"root": root, "levels": levels, "edges": ctx.teps_edges(), "nnz": info["nnz"],
            "active": info["num_active"], "loops": info["num_self_loops"], "max_degree": info["max_degree"]}


def _run_validate(st):
    ctx, root = st["ctx"], st["roots"][0]
    ctx.run_bfs(root)
    pred = ctx.get_pred(st["pred"])
    ok, errors, edges = ctx.validate_pred(root, pred)
    return {"ok": ok, "errors": errors, "edges": edges, "levels": ctx.get_levels(st["out"][0])}


def _run_serve(st):
    srv, q = st["server"], st["queries"]
    res, _ = srv.run(q)
    kept = []
    for i in np.flatnonzero(q["keep"]):
        kept.append(srv.levels(res["request"][i], st["sizes"][q["graph"][i]]))
        srv.release(res["request"][i])
    return {"edges": res["edges"], "status": res["status"], "levels": kept}


def run(state):
    return {"search": _run_search, "batch": _run_batch, "build": _run_build, "validate": _run_validate,
            "serve": _run_serve}[state["case"]["kind"]](state)


def work(case):
    """Bytes a pass cannot do without (nothing here is floating point).

    A search reads, per vertex, its row's bounds and one neighbour and writes
    one level; a batch reads the CSR once and writes a level per root and
    vertex; a build writes and reads the 12-byte tuples and writes 4 bytes
    per directed edge and 8 per vertex; a validation reads every edge.
    """
    kind, ef = case["kind"], case["edgefactor"]
    if kind == "serve":
        scales = [int(s) for s in case["scales"].split(",")]
        mean = sum(1 << s for s in scales) / len(scales)
        return {"bytes": case["queries"] * 13.0 * mean, "flops": 0.0}
    n = float(1 << case["scale"])
    search = 13.0 * n
    if kind == "search":
        return {"bytes": case["roots"] * search, "flops": 0.0}
    if kind == "batch":
        return {"bytes": 8.0 * n * ef + 8.0 * n + case["roots"] * n, "flops": 0.0}
    if kind == "build":
        m = n * ef - case["drop"] + (n - 1 if case["source"] == "spec2012" else 0)
        read = 12.0 * m if case["source"] == "host" else 24.0 * m
        return {"bytes": read + 8.0 * m + 8.0 * n + search, "flops": 0.0}
    return {"bytes": search + 8.0 * n * ef + 8.0 * n + 16.0 * n, "flops": 0.0}


def exact(case, seed):
    """Every output is a whole number, equal on every run: none is a computed floating value."""
    return None

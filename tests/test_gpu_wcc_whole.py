"""WCC by whole-graph pulls: nodes at the edges of the thread, wave and workgroup classes, round limits,
and batches whose instances stop by their own rule, against the oracle and the pushed rounds."""
from ctypes import c_uint64

import numpy as np
import pytest

import mnmgdatalog_amd as dlg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = dlg.Ctx(0)
    yield c
    c.close()


def same(a, b):
    assert (a["iterations"], a["output_size"], a["secondary"]) == (b["iterations"], b["output_size"], b["secondary"])
    assert np.array_equal(a["rows"], b["rows"])


def stars(degrees, seed):
    """Hubs of the given degrees (distinct leaves, some shared between neighbouring hubs), ids shuffled."""
    r, at = [], len(degrees)
    for h, d in enumerate(degrees):
        r.append(np.stack([np.full(d, h), np.arange(at, at + d)], 1))
        at += d - (h % 2)
    r = np.concatenate(r)
    return np.random.default_rng(seed).permutation(r.max() + 1).astype(np.int32)[r]


@pytest.mark.parametrize("degrees", [[1], [15, 16, 17], [16] * 40 + [17] * 40, [1023, 1024, 1025], [8191, 8192, 8193],
                                     [1025, 3, 20_000, 64, 16_384, 16_385, 17]])
def test_degree_classes(ctx, orc, degrees):
    rows = stars(degrees, len(degrees))
    same(ctx.run("wcc", rows), orc.wcc(rows))


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 700])
def test_paths(ctx, orc, n):
    rows = np.stack([np.arange(n), np.arange(1, n + 1)], 1).astype(np.int32)
    same(ctx.run("wcc", rows), orc.wcc(rows))


@pytest.mark.parametrize("k", [1, 2, 3, 4, 7])
def test_truncated(ctx, k):
    rows = np.concatenate([dlg.gen_grid(30, 0.55, 0.01, 20, 3), stars([2000, 9000], 2) + 5000])
    same(ctx.run("wcc", rows, max_iterations=k), ctx.run("wcc", rows, max_iterations=k, strategy=2))


@pytest.mark.parametrize("limit", [0, 1, 3, 6])
def test_batch_stops_each_by_its_own_rule(ctx, limit):
    """Paths (many rounds), stars (few, with hub segments), grids and empty instances side by side."""
    inst = [np.stack([np.arange(w), np.arange(1, w + 1)], 1).astype(np.int32) for w in (1, 5, 60, 300)]
    inst += [stars([17, 16], 1), stars([1500], 2), stars([20_000, 9], 3), np.zeros((0, 2), np.int32)]
    inst += [dlg.gen_grid(24, 0.55, 0.01, 20, s) for s in range(3)]
    kw = {"max_iterations": limit} if limit else {}
    res, _ = ctx.batch_run("wcc", inst, **kw)
    for r, rows in zip(res, inst):
        want = ctx.run("wcc", rows, strategy=2, **kw)
        if len(rows) == 0:
            assert r["output_size"] == 0
            continue
        same(r, want)
        assert r["nodes"] == want["nodes"]


# one workgroup's rounds: the largest it takes and the first it does not (by edges, by nodes), stars, and stops after k rounds
@pytest.mark.parametrize("kind,n", [("path", 15), ("path", 1023), ("path", 1025), ("path", 8192), ("path", 8193), ("star", 1), ("star", 4000),
                                    ("star", 8192), ("star", 8194), ("random", 500), ("random", 8191), ("random", 8192), ("random", 8193),
                                    ("loops", 500), ("loops", 16_384), ("loops", 16_385)])
@pytest.mark.parametrize("k", [1, 2, 6])
def test_one_workgroup(ctx, orc, kind, n, k):
    rng = np.random.default_rng(n)
    if kind == "path":
        rows = np.stack([np.arange(n), np.arange(1, n + 1)], 1)
    elif kind == "star":
        rows = np.stack([np.full(n, n // 2), np.arange(n)], 1)
    elif kind == "random":   # n undirected edges, each once
        a, b = np.triu_indices(1500, 1)
        pick = rng.choice(len(a), n, replace=False)
        rows = np.stack([a[pick], b[pick]], 1)
    else:
        rows = np.stack([np.arange(n), np.arange(n)], 1)
    rows = (rng.permutation(rows.max() + 1)[rows] if kind != "path" else rows).astype(np.int32) - 700
    same(ctx.run("wcc", rows, max_iterations=k), ctx.run("wcc", rows, max_iterations=k, strategy=2))
    if k == 6 and (kind != "path" or n < 2000):
        same(ctx.run("wcc", rows), orc.wcc(rows))


# Few nodes lowered for many rounds in a graph whose pulls cost more than that: the rounds go on by pushes; and back
# to pulls where many nodes are lowered again.
def tail(core, n):
    v = int(core.max()) + 1
    k = np.arange(n)
    return np.concatenate([core, np.stack([np.where(k == 0, core.min(), v + k - 1), v + k], 1)]).astype(np.int32)


def comb(chains, length, gap, feeder):
    """`chains` chains at a hub, which settle in `length` rounds; `gap` rounds after the first the hub sees a lower label
    in each of `feeder` rounds, and so does every chain.  A path beside them has a node fewer to lower in every round, so
    that no two rounds lower as many."""
    hub, g0 = feeder, feeder + 1 + chains * length                       # ids: the feeder, the hub, the chains, the gap
    k = np.arange(chains * length)
    up = np.where(k % length == 0, hub, hub + k)
    path = np.concatenate([np.arange(feeder), g0 + np.arange(gap), [hub]])
    beside = g0 + gap + np.arange(gap + 2 * feeder)
    return np.concatenate([np.stack([path[:-1], path[1:]], 1), np.stack([up, hub + 1 + k], 1),
                           np.stack([beside[:-1], beside[1:]], 1)]).astype(np.int32)


@pytest.fixture(scope="module")
def long_graphs():
    return {"tail": tail(dlg.gen_rmat(17, 2 << 20, 0.57, 0.19, 0.19, 5), 300), "comb": comb(200_000, 40, 200, 100)}


@pytest.mark.parametrize("shape", ["tail", "comb"])
@pytest.mark.parametrize("k", [0, 5, 48, 50, 53, 57, 64, 70, 100, 205, 240, 250, 299])
def test_few_nodes_left(ctx, long_graphs, shape, k):
    rows = long_graphs[shape]
    kw = {"max_iterations": k} if k else {}
    got = ctx.run("wcc", rows, **kw)
    same(got, ctx.run("wcc", rows, strategy=2, **kw))
    if not k:
        same(got, ctx.run("wcc", rows, strategy=1))


@pytest.mark.parametrize("k", [0, 3, 20, 21, 25, 200])
def test_few_nodes_left_batch(ctx, k):
    """A batch of 20M edges, which a pull takes longer for than a pushed round of few nodes: instances that stop before,
    at, and long after the change."""
    rng = np.random.default_rng(1)
    inst = [tail(dlg.gen_rmat(20, 10 << 20, 0.57, 0.19, 0.19, 5), 150), np.array([[5, 4]], np.int32),
            np.stack([np.arange(400), np.arange(1, 401)], 1).astype(np.int32), np.zeros((0, 2), np.int32),
            rng.integers(0, 1000, (1500, 2)).astype(np.int32), tail(dlg.gen_grid(30, 0.55, 0.01, 20, 3), 40)]
    kw = {"max_iterations": k} if k else {}
    res, st = ctx.batch_run("wcc", inst, **kw)
    for r, rows in zip(res, inst):
        if len(rows):
            same(r, ctx.run("wcc", rows, strategy=2, **kw))


def test_pushes_short_of_memory():
    """A resident graph of many nodes to an edge, whose query has memory for pulls but not for the pushed rounds' lists."""
    rows = comb(200_000, 40, 200, 100)
    with dlg.Server(0, workers=1, hbm_budget=8 << 30, retain_bytes=1) as srv:
        g = srv.add_graph(rows)
        free = srv.wait(srv.submit("wcc", graph=g))
    with dlg.Ctx(0) as ctx:
        want = ctx.run("wcc", rows, strategy=2)
        d = ctx.upload(rows)
        for mb in range(900, 2000, 50):   # the graph's build takes most; each is out of memory, or right
            ctx.L.dlg_test_budget(ctx.h, c_uint64(mb << 20))
            try:
                same(ctx.run("wcc", None, device_rows=d, n=len(rows)), want)
            except dlg.DlgError as e:
                assert e.status == dlg.DLG_OUT_OF_MEMORY
        ctx.L.dlg_test_budget(ctx.h, c_uint64(0))
        ctx.free(d)
    assert free["status"] == 0 and free["attempts"] == 1
    same(free, want)

"""TC by row ORs (id ranges up to 2^14 ids): the relation, round count and join rows at the edges of its
words, chunks, tasks and long-list rows, against the oracle and the row kernel (which `queue` selects)."""
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
    assert (a["iterations"], a["output_size"]) == (b["iterations"], b["output_size"])
    assert np.array_equal(a["rows"], b["rows"])


def graph(width, edges, seed, hub=0):
    """`edges` random edges over exactly `width` ids (both ends used), duplicates and self-loops among
    them, the last `hub` ids all pointing at id 3."""
    rng = np.random.default_rng(seed)
    r = rng.integers(0, width, size=(edges, 2))
    r = np.concatenate([r, r[:5], [[0, width - 1], [7 % width, 7 % width]]])
    if hub:
        r = np.concatenate([r, np.stack([np.arange(width - hub, width), np.full(hub, 3)], 1)])
    return (r + rng.integers(-2**30, 2**30)).astype(np.int32)


# words (32), uint4s (128), chunks (2,048) and their remainders; one task to thousands
@pytest.mark.parametrize("width,edges", [(1, 1), (2, 3), (31, 40), (32, 40), (33, 50), (127, 160), (128, 160), (129, 200),
                                         (2047, 2300), (2048, 2300), (2049, 2300), (4097, 4300)])
def test_widths(ctx, orc, width, edges):
    rows = graph(width, edges, width)
    got = ctx.run("tc", rows)
    same(got, orc.tc(rows))
    assert got["raw_join_rows"] == ctx.run("tc", rows, queue=1)["raw_join_rows"]


# the widest range taken, and the first one that is not; several chunks a row, sparse
@pytest.mark.parametrize("width", [16383, 16384, 16385])
def test_widest(ctx, orc, width):
    rows = graph(width, 9000, width)
    got = ctx.run("tc", rows)
    same(got, orc.tc(rows))
    assert got["raw_join_rows"] == ctx.run("tc", rows, queue=1)["raw_join_rows"]


# 255 to 257 and thousands of predecessors: a sub-group's row, then a workgroup's
@pytest.mark.parametrize("hub", [250, 256, 257, 300, 2500])
def test_long_lists(ctx, orc, hub):
    rows = graph(3000, 3500, hub, hub=hub)
    got = ctx.run("tc", rows)
    same(got, orc.tc(rows))
    assert got["raw_join_rows"] == ctx.run("tc", rows, queue=1)["raw_join_rows"]


@pytest.mark.parametrize("k", [1, 2, 3, 5, 9])
def test_truncated(ctx, orc, k):
    rows = graph(700, 760, 11)
    got, want = ctx.run("tc", rows, max_iterations=k), orc.tc(rows, max_iterations=k)
    same(got, want)
    assert got["raw_join_rows"] == ctx.run("tc", rows, queue=1, max_iterations=k)["raw_join_rows"]


def test_many_rounds(ctx, orc):
    rows = np.stack([np.arange(300), np.arange(1, 301)], 1).astype(np.int32)
    got = ctx.run("tc", rows)
    same(got, orc.tc(rows))
    assert got["iterations"] == 300


def test_batch_of_mixed_widths(ctx, orc):
    """One id to several chunks a row, long lists, empty and single-edge instances side by side: each
    as its plain run, with and without a round limit."""
    inst = [graph(w, w + w // 8 + 1, w, hub=h) for w, h in ((1, 0), (33, 0), (640, 400), (129, 0), (2600, 0), (5000, 300))]
    inst.insert(2, np.zeros((0, 2), np.int32))
    inst.append(np.array([[5, 6]], np.int32))
    for kw in ({}, {"max_iterations": 3}):
        res, _ = ctx.batch_run("tc", inst, **kw)
        for r, rows in zip(res, inst):
            same(r, orc.tc(rows, **kw))


@pytest.mark.parametrize("prog", ["tc", "wcc"])
def test_batch_digest_segments(ctx, prog):
    """Instances of one tuple to several of the digest's segments of 2^15 tuples, and empty ones
    between them: each instance's digest is its plain run's."""
    sizes = [1, 0, 181, 182, 2, 0, 0, 300, 33] if prog == "tc" else [1, 40_000, 0, 2, 70_000]
    inst = []
    for i, w in enumerate(sizes):   # a cycle of w ids: w * w tuples; w self-loops: w components
        k = np.arange(w)
        inst.append((np.stack([k, (k + 1) % max(w, 1) if prog == "tc" else k], 1) + 100 * i).astype(np.int32))
    res, _ = ctx.batch_run(prog, inst, keep_output=False, check_output=1)
    for r, rows in zip(res, inst):
        p = ctx.run(prog, rows, keep_output=False, check_output=1)
        assert (r["output_size"], r["output_sum"]) == (p["output_size"], p["output_sum"])
        assert r["output_order_breaks"] == p["output_order_breaks"] == 0


# one workgroup's closure: the widest ranges it takes and the first it does not (by the map, by the edges' lists, by
# their number), many rounds, a hub, duplicates, and stops after k rounds
@pytest.mark.parametrize("width,edges", [(128, 8185), (129, 8186), (384, 400), (385, 400), (512, 600), (640, 700), (640, 8000), (697, 1200),
                                         (704, 2500), (720, 900), (735, 750), (768, 800), (769, 800), (1024, 1100)])
@pytest.mark.parametrize("k", [0, 3])
def test_one_workgroup(ctx, orc, width, edges, k):
    rows = graph(width, edges, width + edges, hub=width // 3)
    rows = rows[:8192] if edges == 8185 else rows
    kw = {"max_iterations": k} if k else {}
    got = ctx.run("tc", rows, **kw)
    same(got, orc.tc(rows, **kw))
    assert got["raw_join_rows"] == ctx.run("tc", rows, queue=1, **kw)["raw_join_rows"]


@pytest.mark.parametrize("n", [1, 300, 700])
@pytest.mark.parametrize("k", [0, 1, 2, 5])
def test_one_workgroup_paths(ctx, orc, n, k):
    rows = np.stack([np.arange(n), np.arange(1, n + 1)], 1)
    rows = np.concatenate([rows, rows[:7], rows[:7]]).astype(np.int32) - 2**31 // 2
    kw = {"max_iterations": k} if k else {}
    got = ctx.run("tc", rows, **kw)
    same(got, orc.tc(rows, **kw))
    assert got["raw_join_rows"] == ctx.run("tc", rows, queue=1, **kw)["raw_join_rows"]


@pytest.mark.parametrize("hubs", [1, 7, 8, 9, 20])
@pytest.mark.parametrize("k", [0, 2])
def test_one_workgroup_hubs(ctx, orc, hubs, k):
    """Rows of 128 to 130 predecessors and more: those that one workgroup shares, and more of them than it takes."""
    r = [np.stack([np.arange(128 + h % 3 + 9 * (h == 4)), np.full(128 + h % 3 + 9 * (h == 4), 200 + h)], 1) for h in range(hubs)]
    rows = np.concatenate(r + [np.stack([np.arange(300, 420), np.arange(301, 421)], 1), [[200, 300], [200 + hubs - 1, 5], [420, 7]]]).astype(np.int32)
    kw = {"max_iterations": k} if k else {}
    got = ctx.run("tc", rows, **kw)
    same(got, orc.tc(rows, **kw))
    assert got["raw_join_rows"] == ctx.run("tc", rows, queue=1, **kw)["raw_join_rows"]


def budget(ctx, mb):
    ctx.L.dlg_test_budget(ctx.h, c_uint64(int(mb * (1 << 20))))


# 16,384 ids: maps of 32 MB, the row ORs' three in 96; the row kernel's one and its copy for the read-out in 64.  With
# small ranges beside it a map is a little larger, in blocks of 40 MB (the pool's size class): 120 and 80.
@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("mb", [1, 8, 31, 33, 50, 65, 80, 95, 97, 99, 128])
def test_short_of_memory(ctx, orc, batch, mb):
    inst = [graph(16384, 9000, 1)] if not batch else [graph(16384, 9000, 1), graph(300, 400, 2), graph(20, 9, 3)]

    def run():
        return ctx.batch_run("tc", inst)[0] if batch else [ctx.run("tc", inst[0])]

    budget(ctx, mb)
    try:
        got = run()
    except dlg.DlgError as e:
        assert e.status == dlg.DLG_OUT_OF_MEMORY and mb < (95 if batch else 80)
        got = None
    finally:
        budget(ctx, 0)
    for g in (got, run()):   # and what follows it
        for r, rows in zip(g or [], inst):
            same(r, orc.tc(rows))
            if not batch:
                assert r["raw_join_rows"] == ctx.run("tc", rows, queue=1)["raw_join_rows"]


# many small instances: maps in tiles of 256 words where those of 2,048 would mostly pad, in fewer and in more tiles than
# CUs take (256 x 2,048 words), one map of several tiles among them
@pytest.mark.parametrize("count,ids", [(1, 10), (5, 64), (300, 30), (3000, 12), (3000, 70), (40, 200)])
def test_many_small_instances(ctx, orc, count, ids):
    rng = np.random.default_rng(count + ids)
    inst = [rng.integers(-ids, ids, size=(ids // 2, 2)).astype(np.int32) // 2 for _ in range(count)]
    inst.append(graph(150, 170, 9))
    res, _ = ctx.batch_run("tc", inst, check_output=1)
    for r, rows in zip(res, inst):
        want = orc.tc(rows)
        same(r, want)
        assert r["output_order_breaks"] == 0


def test_tiny_instances_memory(ctx):
    """20,000 instances of up to 10 ids in 256 MB (the maps in tiles of 2,048 words: three of 160)."""
    rng = np.random.default_rng(2)
    inst = [rng.integers(0, 10, size=(8, 2)).astype(np.int32) for _ in range(20_000)]
    want, _ = ctx.batch_run("tc", inst, keep_output=False, check_output=1)
    row_kernel, _ = ctx.batch_run("tc", inst, keep_output=False, check_output=1, queue=1)
    assert want == row_kernel
    budget(ctx, 256)
    try:
        assert ctx.batch_run("tc", inst, keep_output=False, check_output=1)[0] == want
    finally:
        budget(ctx, 0)

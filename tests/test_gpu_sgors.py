"""SG by two row ORs (id ranges whose map a 32-bit byte offset covers): the relation, round count and join rows at the edges of
its words, tiles, chunks and long-list rows, against the oracle and the sorted lists (`strategy=1`)."""
import numpy as np
import pytest

import mnmgdatalog_amd as dlg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = dlg.Ctx(0)
    yield c
    c.close()


def check(ctx, want, rows, **kw):
    got, lists = ctx.run("sg", rows, **kw), ctx.run("sg", rows, strategy=1, **kw)
    for r in (want, lists):
        assert (got["iterations"], got["output_size"]) == (r["iterations"], r["output_size"])
        assert np.array_equal(got["rows"], r["rows"])
    assert got["raw_join_rows"] == lists["raw_join_rows"]


def graph(width, edges, seed, hub=0, near=0):
    """`edges` random edges over exactly `width` ids, of ends within `near` of each other if given,
    duplicates and self-loops among them; `hub` ids spread over the range all pointing at id 3."""
    rng = np.random.default_rng(seed)
    r = rng.integers(0, width, size=(edges, 2))
    if near:
        r[:, 1] = np.minimum(width - 1, r[:, 0] + rng.integers(1, near, size=edges))
    r = np.concatenate([r, r[:5], [[0, width - 1], [7 % width, 7 % width]]])
    if hub:
        r = np.concatenate([r, np.stack([np.linspace(0, width - 1, hub).astype(np.int64), np.full(hub, 3)], 1)])
    return (r + rng.integers(-2**30, 2**30)).astype(np.int32)


# words (32), uint4s (128), tiles of 512 rows, chunks (1,024) and their remainders
@pytest.mark.parametrize("width,edges", [(1, 1), (2, 3), (31, 40), (32, 40), (33, 50), (63, 70), (65, 70), (127, 160), (128, 160),
                                         (129, 200), (511, 600), (512, 600), (513, 600), (1023, 1100), (1024, 1100), (1025, 1100), (2049, 2200)])
def test_widths(ctx, orc, width, edges):
    rows = graph(width, edges, width)
    check(ctx, orc.sg(rows), rows)


# groups of 8 chunks (8,192 ids) and their remainders
@pytest.mark.parametrize("width", [8191, 8192, 8193, 16385, 17409, 65537])
def test_tiles(ctx, orc, width):
    rows = graph(width, 9000, width, near=40)
    check(ctx, orc.sg(rows), rows)


# the widest range taken, and the first one that is not
@pytest.mark.parametrize("width", [185344, 185345])
def test_widest(ctx, orc, width):
    rows = graph(width, 60000, width, near=40)
    check(ctx, orc.sg(rows), rows)


# 8, 9, 64, 65 and thousands of predecessors: one reading, two, then all of a workgroup's waves
@pytest.mark.parametrize("width,hub", [(3000, 8), (3000, 9), (3000, 60), (3000, 64), (3000, 66), (3000, 1500), (17000, 300)])
def test_long_lists(ctx, orc, width, hub):
    rows = graph(width, width // 2, hub, hub=hub, near=9)
    check(ctx, orc.sg(rows), rows)


@pytest.mark.parametrize("k", [1, 2, 3, 5, 9])
def test_truncated(ctx, orc, k):
    rows = graph(700, 760, 11)
    check(ctx, orc.sg(rows, max_iterations=k), rows, max_iterations=k)


def test_many_rounds(ctx, orc):
    """A ladder: a round finds the pairs one rung further on."""
    k = np.arange(400)
    rows = np.concatenate([np.stack([2 * k, 2 * k + 2], 1), np.stack([2 * k + 1, 2 * k + 3], 1), [[0, 1]]]).astype(np.int32)
    check(ctx, orc.sg(rows), rows)


def test_no_pairs(ctx, orc):
    rows = np.array([[1, 2], [3, 4], [4, 4]], np.int32)   # the base rule gives nothing
    check(ctx, orc.sg(rows), rows)

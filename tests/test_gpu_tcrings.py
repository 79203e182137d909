"""TC over exactly symmetric graphs of small degree by lists of words: the relation, round count and join
rows against the row kernel (which `queue` selects) and, where it is small, the oracle."""
import numpy as np
import pytest

import mnmgdatalog_amd as dlg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = dlg.Ctx(0)
    yield c
    c.close()


def both(rows):
    return np.concatenate([rows, rows[:, ::-1]]).astype(np.int32)


def check(ctx, rows, oracle=None, **kw):
    got, want = ctx.run("tc", rows, **kw), ctx.run("tc", rows, queue=1, **kw)
    for k in ("iterations", "output_size", "raw_join_rows"):
        assert got[k] == want[k]
    assert np.array_equal(got["rows"], want["rows"])
    if oracle:
        o = oracle(rows, **{k: v for k, v in kw.items() if k == "max_iterations"})
        assert (got["iterations"], got["output_size"]) == (o["iterations"], o["output_size"])
        assert np.array_equal(got["rows"], o["rows"])


def forest(width, parts, seed, extra=0):
    """Symmetric edges over exactly `width` ids: paths of random lengths, `extra` more edges within
    near ids, self-loops and repeated edges."""
    rng = np.random.default_rng(seed)
    name = rng.permutation(width)
    name[[0, width - 1]] = 0, width - 1   # both ends of the range are used
    k = np.arange(width - 1)
    k = k[np.isin(k, rng.choice(width - 1, parts, replace=False), invert=True)]
    r = np.stack([name[k], name[k + 1]], 1)
    if extra:
        a = rng.integers(0, width - 9, size=extra)
        r = np.concatenate([r, np.stack([name[a], name[a + rng.integers(1, 9, size=extra)]], 1)])
    r = np.concatenate([r, r[:4], [[0, 0], [width - 1, width - 1]], np.stack([name[:3], name[:3]], 1)])
    return both(r) + np.int32(rng.integers(-2**30, 2**30))


# the first range taken, word and wave remainders; hundreds of short paths
@pytest.mark.parametrize("width", [16385, 16391, 16415, 20000, 33001])
def test_widths(ctx, orc, width):
    check(ctx, forest(width, 600, width), orc.tc)


# degrees up to 8 and past it (9: the row kernel's), lists of all eight neighbours
@pytest.mark.parametrize("degree", [1, 4, 5, 7, 8, 9])
def test_degrees(ctx, orc, degree):
    hubs = np.arange(0, 17000, 20)
    r = np.concatenate([np.stack([hubs, hubs + 1 + d], 1) for d in range(degree)] + [[[17100, 17101]]])
    check(ctx, both(r), orc.tc)


@pytest.mark.parametrize("k", [1, 2, 3, 62, 63, 64, 65, 70])
def test_truncated(ctx, k):
    """Around the 64 rounds that a list buffer holds, too."""
    check(ctx, forest(17000, 60, 5), max_iterations=k)


def test_many_rounds(ctx):
    check(ctx, forest(16500, 40, 6))   # paths of hundreds of ids: several buffers' worth of rounds


@pytest.mark.parametrize("side,p", [(131, 0.62), (140, 1.0)])
def test_full_buffers(ctx, side, p):
    """Rings of hundreds of words a source (lists of more than the 512 entries in flight on the whole
    grid): the buffers fill before 64 rounds."""
    check(ctx, dlg.gen_grid(side, p, 0.0, 20, side))


def test_one_edge_short_of_symmetric(ctx, orc):
    check(ctx, forest(17000, 600, 8)[1:], orc.tc)   # not taken


def test_no_room_for_the_lists(orc):
    """A memory budget that holds F (36 MB) but not the lists beside it: the row kernel's run."""
    rows = forest(17000, 2500, 9)
    want = orc.tc(rows)
    with dlg.Server(0, workers=1, hbm_budget=256 << 20, retain_bytes=1) as srv:
        got = srv.wait(srv.submit("tc", rows))
    assert (got["iterations"], got["output_size"]) == (want["iterations"], want["output_size"])
    assert np.array_equal(got["rows"], want["rows"])


@pytest.mark.parametrize("width", [16_400, 20_000])
@pytest.mark.parametrize("k", [0, 1, 2, 3, 4, 5])
def test_few_large_rings(ctx, width, k):
    """Random neighbours, eight of them: the rings reach most words in a few rounds.  The first buffer has wpr / 4 entries a
    source (wpr words a row) and takes the rounds of 8 and 56 ends; the second, four times as large, does not take the next
    two (392 ends in 54 % of the words, 2,744 in nearly all): the run starts again with buffers for two rounds of any size."""
    rng = np.random.default_rng(width)
    rows = both(np.concatenate([np.stack([np.arange(width), rng.permutation(width)], 1) for _ in range(4)]))
    kw = {"keep_output": False, "check_output": 1, **({"max_iterations": k} if k else {})}
    got, want = ctx.run("tc", rows, **kw), ctx.run("tc", rows, queue=1, **kw)
    for f in ("iterations", "output_size", "raw_join_rows", "output_sum", "output_order_breaks"):
        assert got[f] == want[f]
    if not k:
        assert got["output_size"] == width * width


# the widest range taken, and the first one that is not
@pytest.mark.parametrize("width", [184_319, 184_320, 184_321])
def test_widest(ctx, width):
    check(ctx, forest(width, 6000, width, extra=2000))

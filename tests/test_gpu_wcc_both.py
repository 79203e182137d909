"""WCC inputs that list both directions of their edges, sorted: taken as their own reverse, and the
same relation with one row changed so that it no longer is, against the components of the unsorted rows and the oracle."""
import numpy as np
import pytest

import mnmgdatalog_amd as dlg

pytestmark = pytest.mark.gpu

N = 70_001   # rows, from which on the reverse is looked for (65,536)


@pytest.fixture(scope="module")
def ctx():
    c = dlg.Ctx(0)
    yield c
    c.close()


def in_order(rows):
    return np.unique(rows.astype(np.int32), axis=0)   # by (source, end), no duplicates


def both(rows):
    return in_order(np.concatenate([rows, rows[:, ::-1]]))


def random_rows(n, ids, seed, lo=0):
    return np.random.default_rng(seed).integers(0, ids, (n, 2)) + lo


def check(ctx, orc, rows):
    rows = np.ascontiguousarray(rows, dtype=np.int32)
    got, want = ctx.run("wcc", rows), orc.wcc(rows)
    assert (got["iterations"], got["output_size"], got["secondary"]) == (want["iterations"], want["output_size"], want["secondary"])
    assert np.array_equal(got["rows"], want["rows"])
    mixed = ctx.run("wcc", np.random.default_rng(1).permutation(rows))
    assert np.array_equal(got["rows"], mixed["rows"]) and got["nodes"] == mixed["nodes"] and got["iterations"] == mixed["iterations"]


@pytest.mark.parametrize("n,ids,lo", [(N, 9000, 0), (N, 200_000, -100_000), (N, 1_000_000, 2**31 - 1_000_000), (600_000, 30_000, -5)])
def test_both_directions(ctx, orc, n, ids, lo):
    check(ctx, orc, both(random_rows(n, ids, n + ids, lo)))


@pytest.mark.parametrize("change", ["one row fewer", "ends moved", "reversed once more", "two rows swapped", "a duplicate", "self-loops",
                                    "one direction"])
def test_one_row_changed(ctx, orc, change):
    rows = both(random_rows(N, 50_000, 5))
    rows = rows[rows[:, 0] != rows[:, 1]]
    k = len(rows) // 3
    if change == "one row fewer":
        rows = np.delete(rows, k, 0)
    elif change == "ends moved":   # the only row of a new id: its node and its edge come by the reverse
        rows = in_order(np.concatenate([np.delete(rows, k, 0), [[rows[k, 0], 60_000]]]))
    elif change == "reversed once more":
        rows = in_order(np.concatenate([rows, [[rows[k, 0], 70_000], [80_000, rows[k, 1]]]]))
    elif change == "two rows swapped":
        rows[[k, k + 1]] = rows[[k + 1, k]]
    elif change == "a duplicate":
        rows = np.insert(rows, k, rows[k], 0)
    elif change == "self-loops":
        rows = in_order(np.concatenate([rows, [[3, 3], [90_000, 90_000]]]))
    else:
        rows = rows[rows[:, 0] < rows[:, 1]]
        assert len(rows) >= 2**16
    check(ctx, orc, rows)


@pytest.mark.parametrize("hubs", [1, 3, 700])
def test_pulled_rounds(ctx, orc, hubs):
    """Pushed and pulled rounds: hubs over whole waves and tiles, nodes of one edge, a last tile that is not full."""
    rng = np.random.default_rng(hubs)
    leaf = rng.integers(0, 60_000, 90_000)
    rows = both(np.concatenate([np.stack([leaf % hubs + 60_000, leaf], 1), np.stack([leaf, rng.integers(0, 60_000, 90_000)], 1)]))
    rows = rows + np.int32(-30_000)
    want = orc.wcc(rows)
    for form in (1, 2):
        got = ctx.run("wcc", rows, strategy=1, relax=form)
        assert (got["iterations"], got["output_size"], got["secondary"]) == (want["iterations"], want["output_size"], want["secondary"])
        assert np.array_equal(got["rows"], want["rows"])

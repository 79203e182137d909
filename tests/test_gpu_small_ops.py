"""Operators by one workgroup (up to 8,192 tuples) and the set difference's staged search, at the edges of
their sizes and against numpy; calls whose output overlaps an input."""
import ctypes

import numpy as np
import pytest

import mnmgdatalog_amd as dlg

pytestmark = pytest.mark.gpu
SIZES = [1, 2, 63, 64, 65, 1023, 1024, 1025, 2048, 2049, 4096, 4097, 8191, 8192, 8193, 9000]


@pytest.fixture(scope="module")
def ctx():
    c = dlg.Ctx(0)
    yield c
    c.close()


def tuples(rng, n, kind):
    if kind == "narrow":      # few bits, many duplicates
        hi, lo = rng.integers(5, 25, n), rng.integers(7, 40, n)
    elif kind == "key":       # one value: the value half takes no bits
        hi, lo = rng.integers(0, 1 << 20, n), np.full(n, 9)
    elif kind == "equal":
        hi, lo = np.full(n, 3), np.full(n, 4)
    else:                     # every bit, the extremes among them
        hi, lo = rng.integers(0, 1 << 32, n), rng.integers(0, 1 << 32, n)
        hi[: min(n, 2)] = [0, (1 << 32) - 1][: min(n, 2)]
        lo[: min(n, 2)] = [0, (1 << 32) - 1][: min(n, 2)]
    return (hi.astype(np.uint64) << np.uint64(32)) | lo.astype(np.uint64)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("kind", ["wide", "narrow", "key", "equal"])
def test_sort_unique(ctx, n, kind):
    t = tuples(np.random.default_rng(n), n, kind)
    assert np.array_equal(ctx.sort(t), np.sort(t))
    assert np.array_equal(ctx.sort_unique(t), np.unique(t))


@pytest.mark.parametrize("n", [1, 255, 1024, 1025, 8192, 8193, 20_000])
def test_hash_join_small(ctx, n):
    """The index built by one workgroup: every (probe, row) pair once."""
    rng = np.random.default_rng(n)
    rel = dlg.pack(rng.integers(0, max(2, n // 3), (n, 2)).astype(np.int32))
    probe = dlg.pack(rng.integers(0, max(2, n // 3), (50, 2)).astype(np.int32))
    got, info = ctx.hash_join(rel, probe)
    r, p = dlg.unpack(rel), dlg.unpack(probe)
    want = np.array([(v, pv) for pk, pv in p for v in r[r[:, 0] == pk][:, 1]], np.int32).reshape(-1, 2)
    assert np.array_equal(np.sort(got), np.sort(dlg.pack(want)))
    assert (info["rows"], info["keys"]) == (n, len(np.unique(r[:, 0])))


# tiles of 2,048 in parts of 512; stretches of `other` of none to thousands per part, staged or not
@pytest.mark.parametrize("na", [1, 511, 512, 513, 2048, 8191, 8192, 8193, 8704, 10_241, 40_000])
@pytest.mark.parametrize("nb", [1, 1023, 1025, 9000, 300_000])
def test_set_difference(ctx, na, nb):
    rng = np.random.default_rng(na * 7 + nb)
    pool = np.unique(rng.integers(0, 1 << 63, na + nb, dtype=np.uint64))
    a = np.unique(rng.choice(pool, na))
    b = np.unique(np.concatenate([rng.choice(pool, nb), a[:: 3]]))
    assert np.array_equal(ctx.set_difference(a, b), np.setdiff1d(a, b))


@pytest.mark.parametrize("na,nb", [(100, 50), (9000, 20_000)])
def test_set_difference_clustered(ctx, na, nb):
    """All of `other` inside one part's range, or outside every part's."""
    a = np.arange(na, dtype=np.uint64) * np.uint64(1 << 40)
    inside = np.arange(1, nb + 1, dtype=np.uint64) + a[na // 2]
    for b in (inside, np.append(inside, a[na // 2 + 1]), inside + a[-1], np.array([0], np.uint64)):
        assert np.array_equal(ctx.set_difference(a, np.unique(b)), np.setdiff1d(a, b))


@pytest.mark.parametrize("n", [500, 30_000])
@pytest.mark.parametrize("where", ["a", "b", "inside a", "apart"])
def test_set_difference_output_place(ctx, n, where):
    rng = np.random.default_rng(n)
    a = np.unique(rng.integers(0, 4 * n, n).astype(np.uint64))
    b = np.unique(rng.integers(0, 4 * n, n).astype(np.uint64))
    room_after = np.zeros(len(a), np.uint64)
    pa, pb = ctx.upload(np.concatenate([a, room_after])), ctx.upload(np.concatenate([b, room_after]))
    room = ctx.alloc(8 * (len(a) + len(b)))
    out = {"a": pa, "b": pb, "inside a": pa + 8 * (len(a) // 2), "apart": room}[where]
    k = ctypes.c_int64()
    ctx.check(ctx.L.dlg_set_difference(ctx.h, pa, len(a), pb, len(b), out, ctypes.byref(k)), "set_difference")
    assert np.array_equal(ctx.download(out, k.value, np.uint64), np.setdiff1d(a, b))
    for p in (pa, pb, room):
        ctx.free(p)

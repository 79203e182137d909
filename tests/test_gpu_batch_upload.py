"""Batches whose rows are bounded and shifted on the device: totals around the first that is (65,536 rows), empty
instances, instances over several chunks of the upload (262,144 rows) and segments (4,096), ids at both ends of their range."""
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


def check(ctx, prog, inst):
    res, _ = ctx.batch_run(prog, inst, check_output=1)
    for r, rows in zip(res, inst):
        if len(rows) == 0:
            assert r["output_size"] == 0
            continue
        want = ctx.run(prog, rows, check_output=1)
        assert (r["iterations"], r["output_size"], r["secondary"]) == (want["iterations"], want["output_size"], want["secondary"])
        assert np.array_equal(r["rows"], want["rows"])
        assert (r["output_sum"], r["output_order_breaks"]) == (want["output_sum"], want["output_order_breaks"])


def rows(n, ids, lo, seed):
    return (np.random.default_rng(seed).integers(0, ids, (n, 2)) + lo).astype(np.int32)


@pytest.mark.parametrize("total", [65_535, 65_536, 65_537])
@pytest.mark.parametrize("prog", ["tc", "wcc"])
def test_first_total(ctx, prog, total):
    inst = [rows(n, n, -n // 2, n) for n in (1, 700, 4096)] + [np.zeros((0, 2), np.int32), rows(255, 200, 5, 1)]
    inst.append(rows(total - sum(len(r) for r in inst), 90_000, -40_000, 2))
    check(ctx, prog, inst)


@pytest.mark.parametrize("prog", ["wcc", "single_join"])
def test_chunks_and_ends(ctx, prog):
    empty = np.zeros((0, 2), np.int32)
    inst = [empty, rows(262_143, 60_000, -2**31, 1), empty, rows(1, 1, 2**31 - 1, 2), rows(262_145, 70_000, 2**31 - 70_000, 3),
            rows(4097, 900, 0, 4), rows(40_000, 5000, -7, 5), empty]
    check(ctx, prog, inst)


@pytest.mark.parametrize("total", [100_000, 524_287, 524_289, 4_000_000])
def test_page_locked(ctx, total):
    """The rows go up by two chunks of 2 MB at most, however many they are."""
    pinned = ctx.L.dlg_test_pinned_bytes
    pinned.restype = c_uint64
    inst = [rows(total // 4, 30_000, 0, k) for k in range(4)]
    before = pinned()
    res, _ = ctx.batch_run("wcc", inst, keep_output=False)
    assert pinned() - before <= 4 << 20
    want = [ctx.run("wcc", i, keep_output=False) for i in inst]
    assert [(r["iterations"], r["output_size"], r["secondary"]) for r in res] == [
        (w["iterations"], w["output_size"], w["secondary"]) for w in want]

"""A batch that fails while its rows go to the host: its blocks, which the next call may be given, are not written
any more once the call has returned."""
import time
from ctypes import byref, c_int64, c_void_p, memset, sizeof

import numpy as np
import pytest

import mnmgdatalog_amd as dlg

pytestmark = pytest.mark.gpu


def cycle(n, at=0):
    k = np.arange(n)
    return (np.stack([k, (k + 1) % n], 1) + at).astype(np.int32)


def closure(n, at=0):
    k = np.arange(n) + at
    return np.stack([np.tile(k, n), np.repeat(k, n)], 1)   # (src, dst) by (dst, src)


def fail_block(n):
    dlg.lib().dlg_test_fail_host_block(c_int64(n))


@pytest.mark.parametrize("count", [2, 65])
def test_block_fails(count):
    """Blocks of 8 MB: the first `count` - 1 are had, their copies (0.5 GB, 9 ms, for 64) would be queued; the last is not."""
    n = 1000
    with dlg.Ctx(0) as ctx, dlg.Ctx(0) as other:
        inst = [cycle(n)] * count
        other.run("tc", cycle(n))   # its pool is warm
        fail_block(count - 1)
        with pytest.raises(dlg.DlgError) as e:
            ctx.batch_run("tc", inst)
        fail_block(-1)
        assert e.value.status == dlg.DLG_OUT_OF_MEMORY
        rows = other.run("tc", cycle(n, 7))["rows"]   # takes a block of the failed call
        time.sleep(0.05)
        assert np.array_equal(rows, closure(n, 7))
        res, _ = ctx.batch_run("tc", inst[:2])        # the context goes on
        for r in res:
            assert np.array_equal(r["rows"], closure(n))


def test_served_batch_fails():
    """A served batch whose second block fails: its requests run again, by themselves, and are right."""
    with dlg.Server(0, workers=1, max_batch=8) as srv:
        first = srv.submit("tc", cycle(3000))   # holds the one slot while the others queue up
        fail_block(3)
        ts = [srv.submit("tc", cycle(40 + i)) for i in range(6)]
        got = [srv.wait(t) for t in [first] + ts]
        fail_block(-1)
    assert all(g["status"] == 0 for g in got)
    for i, g in enumerate(got[1:]):
        assert np.array_equal(g["rows"], closure(40 + i))


@pytest.mark.parametrize("total", [10, 70_000])
def test_results_given_uncleared(total):
    """Results that hold what the caller left in them, and a batch refused before any is filled in: ids that do not fit."""
    inst = [np.array([[-2**31, 2**31 - 1]] * total, np.int32), np.array([[0, 1]], np.int32)]
    with dlg.Ctx(0) as ctx:
        ptrs = (c_void_p * 2)(*[a.ctypes.data for a in inst])
        ns = (c_int64 * 2)(*[len(a) for a in inst])
        res, st, o = (dlg.Result * 2)(), dlg.BatchStats(), dlg.Opts()
        memset(byref(res), 0x5a, sizeof(res))
        s = ctx.L.dlg_batch_run(ctx.h, dlg.PROGS["tc"], 2, ptrs, ns, byref(o), res, byref(st))
        assert s == dlg.DLG_OVERFLOW
        assert all(not r.rows and r.n_rows == 0 for r in res)

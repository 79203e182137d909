"""Result rows in page-locked host blocks that are kept and handed out again: a result held by the caller
keeps its rows whatever runs after it, on several threads too, and with no context left."""
import threading

import numpy as np
import pytest

import mnmgdatalog_amd as dlg

pytestmark = pytest.mark.gpu


def cycle(n, at):
    k = np.arange(n)
    return (np.stack([k, (k + 1) % n], 1) + at).astype(np.int32)


def want(n, at):
    k = np.arange(n) + at
    return np.stack([np.tile(k, n), np.repeat(k, n)], 1)   # (src, dst) by (dst, src)


@pytest.mark.parametrize("n", [1, 11, 200])
def test_held_results_stay(n):
    ctx = dlg.Ctx(0)
    held = [ctx.run("tc", cycle(n, 1000 * i))["rows"] for i in range(4)]
    for i in range(0, 4, 2):
        held[i] = None   # given back: the next runs take these blocks
    again = [ctx.run("tc", cycle(n, 50_000 + 1000 * i))["rows"] for i in range(4)]
    ctx.close()
    for i in (1, 3):
        assert np.array_equal(held[i], want(n, 1000 * i))
    for i in range(4):
        assert np.array_equal(again[i], want(n, 50_000 + 1000 * i))


def test_threads():
    bad = []

    def work(t):
        with dlg.Ctx(0) as ctx:
            for i in range(12):
                n, at = 5 + 17 * ((t + i) % 5), 10_000 * t + 100 * i
                if not np.array_equal(ctx.run("tc", cycle(n, at))["rows"], want(n, at)):
                    bad.append((t, i))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad

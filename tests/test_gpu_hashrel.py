"""TC and SG over wide id ranges: join rows inserted into the hash set as they are formed, against the
oracle and the sorted-run layout (strategy 2)."""
from ctypes import CDLL, byref, c_size_t

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


# tiles of 256 rows and their remainders; the tuple that equals the empty slot marker (INT32_MAX twice)
@pytest.mark.parametrize("prog", ["tc", "sg"])
@pytest.mark.parametrize("edges", [1, 255, 256, 257, 3000])
@pytest.mark.parametrize("lf", [0.0, 0.1, 0.95])
def test_small(ctx, orc, prog, edges, lf):
    rng = np.random.default_rng(edges)
    rows = (rng.integers(0, max(2, edges), size=(edges, 2)) * 100_003).astype(np.int32)
    rows = np.concatenate([rows, rows[:3], [[2**31 - 1, 2**31 - 1], [5, 2**31 - 1]]]).astype(np.int32)
    kw = {"load_factor": lf} if lf else {}
    got = ctx.run(prog, rows, **kw)
    same(got, getattr(orc, prog)(rows))
    assert got["raw_join_rows"] == ctx.run(prog, rows, strategy=2)["raw_join_rows"]


# far more join rows than new tuples (the rows past the set's room wait for it to grow), hubs
@pytest.mark.parametrize("prog", ["tc", "sg"])
def test_many_duplicates(ctx, orc, prog):
    rng = np.random.default_rng(3)
    rows = rng.integers(0, 120, size=(3000, 2))
    rows = np.concatenate([rows, [[0, 1_000_000]]]).astype(np.int32)
    rows[:-1] *= 3001
    got = ctx.run(prog, rows, strategy=3)
    same(got, getattr(orc, prog)(rows))
    assert got["raw_join_rows"] == ctx.run(prog, rows, strategy=2)["raw_join_rows"]


@pytest.mark.parametrize("k", [1, 2, 4])
def test_truncated(ctx, orc, k):
    rows = (np.random.default_rng(8).integers(0, 500, size=(520, 2)) * 4096).astype(np.int32)
    same(ctx.run("tc", rows, max_iterations=k), orc.tc(rows, max_iterations=k))
    same(ctx.run("sg", rows, max_iterations=k), orc.sg(rows, max_iterations=k))


def test_large_rounds(ctx):
    """Rounds of more than 2^19 probes (tiles of 2,048 rows), against the sorted-run layout."""
    rows = dlg.gen_erdos_renyi(900_000, 800_000, 4)
    got, want = ctx.run("tc", rows), ctx.run("tc", rows, strategy=2)
    same(got, want)
    assert got["raw_join_rows"] == want["raw_join_rows"]


# rounds queued ahead: tiles of 256 probes and their remainders, many rounds, a hub whose rows one tile does not take,
# far more join rows than the set has room for, and a stop after k rounds
@pytest.mark.parametrize("shape", ["path 255", "path 300", "path 1000", "hub", "cliques"])
@pytest.mark.parametrize("k", [0, 1, 3, 4])
def test_queued_rounds(ctx, orc, shape, k):
    rng = np.random.default_rng(len(shape))
    if shape.startswith("path"):
        n = int(shape.split()[1])
        rows = np.stack([np.arange(n), np.arange(1, n + 1)], 1)
        rows = np.concatenate([rows, rng.integers(0, n, (n // 8, 2))]) if n == 300 else rows
    elif shape == "hub":   # 300 paths of 2 into a hub of 400 ends, another of 17,000
        rows = np.concatenate([np.stack([np.arange(300) + 10, np.full(300, 1)], 1), np.stack([np.full(400, 1), np.arange(400) + 1000], 1),
                               np.stack([np.full(17_000, 2), np.arange(17_000) + 2000], 1), [[1000, 2], [5, 10]]])
    else:
        rows = np.concatenate([np.stack(np.nonzero(~np.eye(40, dtype=bool)), 1) + 50 * i for i in range(6)] + [[[3, 55], [60, 110]]])
    rows = (rows * 101).astype(np.int32)
    kw = {"max_iterations": k} if k else {}
    got = ctx.run("tc", rows, strategy=3, **kw)
    same(got, orc.tc(rows, **kw))
    assert got["raw_join_rows"] == ctx.run("tc", rows, strategy=2, **kw)["raw_join_rows"]


def test_tight_budget(orc):
    """A request under a memory budget that has room for its rounds one by one, but not for several at once."""
    rows = (np.random.default_rng(4).integers(0, 3000, size=(2900, 2)) * 4096).astype(np.int32)
    want = orc.tc(rows)
    for mb in (256, 320, 512):
        with dlg.Server(0, workers=1, hbm_budget=mb << 20, retain_bytes=1, strategy=3) as srv:
            got = srv.wait(srv.submit("tc", rows))
        assert got["status"] == 0
        same(got, want)


def free_bytes():
    free, total = c_size_t(), c_size_t()
    assert CDLL("libamdhip64.so").hipMemGetInfo(byref(free), byref(total)) == 0   # the library that libdlg.so has loaded
    return free.value


def test_room_by_new_tuples():
    """Rounds of 7 and more times as many join rows as new tuples: the set takes room for its tuples, not for the rows."""
    rows = (np.random.default_rng(6).integers(0, 700, size=(40_000, 2)) * 4096).astype(np.int32)
    with dlg.Ctx(0) as c:
        c.run("tc", rows[:100], keep_output=False, strategy=3)
        free = free_bytes()
        got = c.run("tc", rows, keep_output=False, strategy=3, check_output=1)
        used = free - free_bytes()
        want = c.run("tc", rows, keep_output=False, strategy=2, check_output=1)
    assert got["output_size"] == 490_000 and got["output_sum"] == want["output_sum"]
    assert (got["iterations"], got["raw_join_rows"]) == (want["iterations"], want["raw_join_rows"])
    assert used < 256 << 20


@pytest.mark.parametrize("n,m,seed", [(1159, 2643, 6), (6599, 10_613, 42), (7046, 13_037, 56), (1199, 2767, 69)])
def test_served_within_its_reservation(ctx, n, m, seed):
    """Served closures over a wide id range keep within the memory reserved for them: none is run a second time."""
    ids = np.sort(np.random.default_rng(5).choice(2**31 - 1, n, replace=False)).astype(np.int32)
    rows = ids[np.random.default_rng(seed).integers(0, n, (m, 2))]
    with dlg.Server(0, workers=2, hbm_budget=40 << 30, retain_bytes=1) as srv:
        got = srv.wait(srv.submit("tc", rows))
    assert got["status"] == 0 and got["attempts"] == 1
    same(got, ctx.run("tc", rows, strategy=2))


@pytest.mark.parametrize("prog,ins,outs", [("tc", 3000, 9000), ("tc", 40, 70_000), ("sg", 10, 6000)])
def test_star(ctx, prog, ins, outs):
    """A hub's pairs, nearly all new, from few probes: the set grows past them in a few steps, and the next round, of as many
    rows and none new, begins with the room there is."""
    hub = 7
    rows = np.concatenate([np.stack([100 + np.arange(ins), np.full(ins, hub)], 1),
                           np.stack([np.full(outs, hub), 100 + ins + np.arange(outs)], 1), [[100 + ins, hub]]])
    rows = (rows * 20_011).astype(np.int32)
    kw = {"keep_output": False, "check_output": 1}
    got, want = ctx.run(prog, rows, **kw), ctx.run(prog, rows, strategy=2, **kw)
    for f in ("iterations", "output_size", "raw_join_rows", "output_sum", "output_order_breaks"):
        assert got[f] == want[f]

"""The single join's rows sorted in registers: at the candidate counts where a row takes more registers, or
leaves them for LDS, with empty runs, single runs and repeated values, against the oracle."""
import numpy as np
import pytest

import mnmgdatalog_amd as dlg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = dlg.Ctx(0)
    yield c
    c.close()


@pytest.mark.parametrize("runs", [1, 3, 63, 64, 65])
@pytest.mark.parametrize("count", [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 192, 255, 256, 257, 300])
def test_counts(ctx, orc, runs, count):
    """One row of `count` candidates from `runs` b's (some with none), a hundred times over, the ids
    spread too wide for the map."""
    rng = np.random.default_rng(1000 * runs + count)
    parts = []
    for c in range(100):
        bs = 1000 + c * 70 + np.arange(runs)
        parts.append(np.stack([bs, np.full(runs, c)], 1))                                   # (b, c)
        hi = [40, 300_000][c % 2]                                                           # values often, or rarely, twice
        parts.append(np.stack([100_000 + rng.integers(0, hi, count), rng.choice(bs, count)], 1))   # (a, b)
    parts.append([[399_999, 399_998]])
    rows = np.concatenate(parts).astype(np.int32)
    got, want = ctx.run("single_join", rows, strategy=2), orc.single_join(rows)
    assert got["output_size"] == want["output_size"]
    assert np.array_equal(got["rows"], want["rows"])


@pytest.mark.parametrize("every", [1, 2, 63, 65, 4000])
@pytest.mark.parametrize("n", [1, 3, 255, 256, 257, 5000])
def test_rows_to_sort(ctx, orc, n, every):
    """`n` output rows, every `every`-th of them (and the first) of 300 candidates, which go through LDS, the others of
    two: listed rows at the edges of workgroups, all, few and one of them; one row too long for LDS beside them."""
    rng = np.random.default_rng(7 * n + every)
    c = np.arange(n)
    many = c % every == 0
    a = 10_000 + np.arange(3000)
    b = 20_000 + np.where(many, 0, 1 + c % 50)                     # row c: one b, shared by the rows of many
    parts = [np.stack([b, c], 1), np.stack([rng.choice(a, 300, replace=False), np.full(300, 20_000)], 1)]
    for k in range(50):
        parts.append(np.stack([rng.choice(a, 2, replace=False), np.full(2, 20_001 + k)], 1))
    parts += [[[30_000, n + 1]], np.stack([a, np.full(3000, 30_000)], 1), [[399_999, 399_998]]]
    rows = np.concatenate(parts).astype(np.int32)
    got, want = ctx.run("single_join", rows, strategy=2), orc.single_join(rows)
    assert got["output_size"] == want["output_size"]
    assert np.array_equal(got["rows"], want["rows"])

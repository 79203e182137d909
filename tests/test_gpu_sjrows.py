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
